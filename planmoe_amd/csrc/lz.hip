// GPULZ ("lz") lossless codec for gfx950: byte-identical streams to the reference's
// lz_compress / lz_decompress (custom/compressor/gpulz.cu), built differently.
//
// One wavefront codes one block of 512 symbols (2048 bytes), lane l owning the 8 consecutive
// symbols 8l .. 8l+7:
//   match   every lane keeps the 39 symbols before its last one in registers and tests its 8
//           symbols against their 32-symbol windows (256 compares, no memory traffic).  A
//           position has a match exactly when its symbol occurs in its window; a block where
//           none does is stored as it is.  Otherwise the comparisons are kept as one 32-bit hit
//           mask per position, and the reference's matcher (gpulz.cu:46-85) walks those masks
//           instead of the symbols: a run grows while the next positions hit at the same
//           distance, 8 positions per step.  A block of one repeated value (an empty capacity
//           slot) has a closed form and is not analysed at all.
//   parse   the greedy token walk (gpulz.cu:98-127, one thread there) advances a whole run of
//           literals or one match per step with ballots and scalar bit scans.
//           Runs of one value with nothing else that repeats, as empty slots make between rows, have a closed form too: matches of 1, 2, 4, 8,
//           16 and 32 symbols from their second on.  (Walked, such a block took a wave 20 us: 112 x 2600 with 40 % empty slots 29.8 us to compress,
//           now 12.5 with the launch for the scan that small inputs go without.)
//   pack    token ranks and byte offsets come from one packed wave scan; flags and token bytes
//           are put together in LDS and copied out with aligned word stores.
// The launches (up to 16 MB without the second: a work-group of the placement adds up the sizes before its own itself): sizes of every block (match + parse; two integers and a class byte per block are written, and, of a block
// with matches, its tokens: two bytes a position), an in-place exclusive scan of the sizes by chunks, and
// placement (stored blocks are copied straight through, the tokens of the others packed at
// their final offset; a wave adds up the totals of the chunks before its own, and spare work-groups zero what lies beyond all).  134 MB of N(0, 1):
// 46 + 7 + 54 us; with matches everywhere (half of the values zero) 745 + 7 + 48, and 770 for the placement when it analysed those blocks again.  The reference
// stages every block at a fixed stride in a buffer as large as the input, scans with a library
// call and copies everything once more (gpulz.cu:148-211, 460-494, 220-258); here stored blocks and
// those of one value, all that most buffers are made of, are never staged and no work-group ever waits for another.
#include "common.hpp"

namespace pm {
namespace {

constexpr int LZ_SYMS = 512;             // symbols per block (gpulz.cu:6 / sizeof(float))
constexpr int LZ_WINDOW = 32;            // gpulz.cu:12
constexpr int LZ_BLOCK_BYTES = 2048;
constexpr int LZ_PITCH = WAVE + 4;        // words between a position's masks and the next one's of a lane
constexpr int LZ_WAVES = 8;              // blocks per work-group
constexpr int LZ_SCAN_CHUNK = 8192;      // table entries scanned by one work-group
constexpr int LZ_SUMMED = 8192;          // up to so many blocks the placement adds up the sizes before its own by itself
constexpr int LZ_MAX_CHUNKS = 256;       // (2^31 / 2048 + 1) / 8192 rounded up to the scan's width
constexpr uint32_t NAN_WINDOW = 0x7f800002u;   // key of a NaN seen as a window symbol ...
constexpr uint32_t NAN_AHEAD = 0x7f800001u;    // ... and as a look-ahead symbol: never equal
enum : uint8_t { LZ_STORED = 0, LZ_CONSTANT = 1, LZ_GENERAL = 2 };

// float equality on bit patterns: both zeros share a key, NaNs get a key per role
__device__ __forceinline__ uint32_t window_key(uint32_t bits)
{
    const float f = __uint_as_float(bits);
    const bool is_nan = __builtin_amdgcn_classf(f, 0x003);          // signalling or quiet NaN
    const bool is_zero = __builtin_amdgcn_classf(f, 0x060);         // -0 or +0
    return is_nan ? NAN_WINDOW : (is_zero ? 0u : bits);
}
__device__ __forceinline__ uint32_t ahead_key(uint32_t wkey) { return wkey == NAN_WINDOW ? NAN_AHEAD : wkey; }

// m = 2 * m + (a == b): the comparison lands in the carry, the add-with-carry shifts it in.
// (Written out so that the compiler does not keep these comparisons and the ones of the quick
// any-hit test as one set of 256 live lane masks.)
__device__ __forceinline__ uint32_t shift_in_equal(uint32_t m, uint32_t a, uint32_t b)
{
    // gfx950 wants two wait states between a VALU write of VCC and a VALU read of it
    asm("v_cmp_eq_u32 vcc, %1, %2\n\ts_nop 1\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc"
        : "+v"(m) : "v"(a), "v"(b) : "vcc");
    return m;
}

// 16 bytes at an even address: token bytes start wherever the blocks before them end.  Global
// memory takes such accesses as they are.
typedef pm_u32x4 __attribute__((aligned(2))) lz_u32x4_a2;

// LDS written by some lanes of a wavefront and read by others of the same wavefront
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t wave_exclusive_sum(uint32_t v, uint32_t &total)
{
    uint32_t inc = v;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const uint32_t o = __shfl_up(inc, d, WAVE);
        if (lane_id() >= d) inc += o;
    }
    total = __builtin_amdgcn_readlane(inc, WAVE - 1);
    return inc - v;
}

// what a wavefront knows about its block after the analysis
struct LzBlock {
    uint32_t lens_lo, lens_hi, offs_lo, offs_hi;   // best match per owned position, one byte each
    uint32_t match_mask, start_mask;               // owned positions with a match / that start a token
    uint32_t tok_base, byte_base;                  // tokens and token bytes before this lane
    uint32_t flag_bytes, data_bytes;               // sizes of the block

    // tokens and token bytes before this lane, totals of the block
    __device__ __forceinline__ void count()
    {
        const uint32_t ntok = __popc(start_mask), nmatch = __popc(start_mask & match_mask);
        uint32_t total;
        const uint32_t before = wave_exclusive_sum(ntok | ((4u * ntok - 2u * nmatch) << 16), total);
        tok_base = before & 0xffffu;
        byte_base = before >> 16;
        flag_bytes = ((total & 0xffffu) + 7u) >> 3;
        data_bytes = total >> 16;
    }
    // the tokens that start at the lane's positions, 16 bits each: bit 15 a token, bit 14 a match, its offset - 1 and its length - 1
    __device__ __forceinline__ uint4 tokens() const
    {
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t l = (((i < 4 ? lens_lo : lens_hi) >> (8 * (i & 3))) - 1u) & 0x1fu, o = (((i < 4 ? offs_lo : offs_hi) >> (8 * (i & 3))) - 1u) & 0x1fu;
            const uint32_t t = ((start_mask >> i) & 1u) ? ((match_mask >> i) & 1u ? 0xc000u | (o << 5) | l : 0x8000u) : 0u;
            w[i >> 1] |= t << (16 * (i & 1));
        }
        return make_uint4(w[0], w[1], w[2], w[3]);
    }
};

// 8 consecutive symbols per lane, zero beyond the end of the input
__device__ __forceinline__ void lz_load(const uint32_t *__restrict__ in, int64_t nsym, int64_t block, int lane,
                                        uint32_t (&raw)[8])
{
    const int64_t s0 = block * LZ_SYMS + 8 * lane;
    if (s0 + 8 <= nsym) {
        const uint4 a = *reinterpret_cast<const uint4 *>(in + s0);
        const uint4 b = *reinterpret_cast<const uint4 *>(in + s0 + 4);
        raw[0] = a.x; raw[1] = a.y; raw[2] = a.z; raw[3] = a.w;
        raw[4] = b.x; raw[5] = b.y; raw[6] = b.z; raw[7] = b.w;
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) raw[i] = s0 + i < nsym ? in[s0 + i] : 0u;
    }
}

// Class of the block and, for LZ_GENERAL, everything in `b`.  keys: 544 words of LDS owned by
// the wavefront.  All lanes of the wavefront call it together.
__device__ __forceinline__ int lz_analyse(const uint32_t (&raw)[8], uint32_t *keys, int lane, LzBlock &b)
{
    keys = static_cast<uint32_t *>(__builtin_assume_aligned(keys, 16));
    uint32_t own[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) own[i] = window_key(raw[i]);

    // ---- one repeated value: tokens L (1,1) (2,2) (4,4) (8,8) (16,16) and (32,32) to the end
    const uint32_t first = __builtin_amdgcn_readfirstlane(own[0]);
    uint64_t differ = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) differ |= __ballot(own[i] != first);
    if (first != NAN_WINDOW && differ == 0) {
        b.flag_bytes = 3;
        b.data_bytes = 44;
        return LZ_CONSTANT;
    }

    if (lane < LZ_WINDOW / 4)
        *reinterpret_cast<uint4 *>(keys + 4 * lane) = make_uint4(NAN_WINDOW, NAN_WINDOW, NAN_WINDOW, NAN_WINDOW);
    *reinterpret_cast<uint4 *>(keys + LZ_WINDOW + 8 * lane) = make_uint4(own[0], own[1], own[2], own[3]);
    *reinterpret_cast<uint4 *>(keys + LZ_WINDOW + 8 * lane + 4) = make_uint4(own[4], own[5], own[6], own[7]);
    wave_sync();

    // ---- which positions see their symbol in their window
    uint32_t win[40];                                   // keys[8l .. 8l+39] = positions 8l-32 .. 8l+7
#pragma unroll
    for (int q = 0; q < 10; ++q) {
        const uint4 v = *reinterpret_cast<const uint4 *>(keys + 8 * lane + 4 * q);
        win[4 * q] = v.x; win[4 * q + 1] = v.y; win[4 * q + 2] = v.z; win[4 * q + 3] = v.w;
    }
    // (a lane whose first two symbols are equal, as in every run of ten and more: the masks below are wanted in any case; 2.3 us of a wave on its own)
    uint64_t hit[8];                                    // lane masks, kept in scalar registers
    if (__ballot(ahead_key(own[1]) == own[0]) == 0) {
        uint64_t some = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t k = ahead_key(own[i]);
            hit[i] = 0;
#pragma unroll
            for (int j = 0; j < LZ_WINDOW; ++j) hit[i] |= __ballot(k == win[i + j]);
            some |= hit[i];
        }
        if (some == 0) {                                // 512 literals, 64 zero flag bytes
            wave_sync();                                // the keys may be overwritten by the next block
            b.flag_bytes = LZ_SYMS / 8;
            b.data_bytes = LZ_BLOCK_BYTES;
            return LZ_STORED;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) hit[i] = 1;
    }
    uint32_t live = 0;                                  // positions that some lane has a hit at
#pragma unroll
    for (int i = 0; i < 8; ++i) live |= hit[i] != 0 ? 1u << i : 0u;

    // ---- hit masks: bit j of position 8l+i's = symbol 8l+i equals window symbol 8l+i-32+j.
    // They hold all the matcher needs: while symbol p+r still equals window symbol w+r, bit
    // (w - p + 32) of the mask of position p+r is set.
    // (The positions are a loop, here and in the matcher: written out eight times the code was 15 KB walked once,
    // and a wave alone on its compute unit waited for instructions most of its time.)
    static_assert(8 * LZ_PITCH <= LZ_WINDOW + LZ_SYMS, "the masks take the keys' place");
    uint32_t *hmask = keys;                             // the keys are all in registers by now
    wave_sync();
    // position 8 q + i lies at i * LZ_PITCH + q: the lanes' reads at one distance are neighbours.  Zero behind the block.
    if (lane < 32) hmask[(lane >> 2) * LZ_PITCH + WAVE + (lane & 3)] = 0;
    uint32_t breaks = 0;                                // bit i: symbol 8l+i is not the one before it
#pragma unroll
    for (int i = 0; i < 8; ++i) breaks |= (ahead_key(own[i]) != win[LZ_WINDOW - 1 + i] ? 1u : 0u) << i;
    // A run of one value: q symbols of it lie right before a position.  If a position's hits are those and no others, everywhere, the tokens have a
    // closed form.
    const uint64_t breaking = __ballot(breaks != 0);    // (lane 0: its first symbol)
    const uint64_t lower = breaking & ((1ull << lane) - 1ull), upper = lane < WAVE - 1 ? breaking & ~((2ull << lane) - 1ull) : 0ull;
    const int from = lower ? 63 - __builtin_clzll(lower) : 0, next = upper ? __builtin_ctzll(upper) : 0;
    const uint32_t from_breaks = __shfl(breaks, from), next_breaks = __shfl(breaks, next);
    const int begin = 8 * from + 31 - __builtin_clz(from_breaks | 1u);              // where the run that reaches the lane begins
    const int end = upper ? 8 * next + __builtin_ctz(next_breaks | 256u) : LZ_SYMS;     // and where the one that leaves it ends
    uint32_t others = 0;
    int q = 8 * lane - begin - 1;
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
        uint32_t m = 0;
        if ((live >> i) & 1u) {
            const uint32_t k = ahead_key(win[LZ_WINDOW]);
#pragma unroll
            for (int j = LZ_WINDOW - 1; j >= 0; --j) m = shift_in_equal(m, k, win[j]);
        }
        q = (breaks >> i) & 1u ? 0 : q + 1;
        others |= m ^ (q == 0 ? 0u : q >= 32 ? 0xffffffffu : 0xffffffffu << (32 - q));
        hmask[i * LZ_PITCH + lane] = m;
#pragma unroll
        for (int j = 0; j < 39; ++j) win[j] = win[j + 1];          // the next position's window and symbol
    }
    wave_sync();
    if (__ballot(others != 0) == 0) {
        // a literal, then matches of 1, 2, 4, 8, 16 and 32 symbols, each as far back as it is long, the last one as long as the run is
        uint64_t lens = 0, offs = 0;
        b.start_mask = b.match_mask = 0;
        q = 8 * lane - begin - 1;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            q = (breaks >> i) & 1u ? 0 : q + 1;
            const uint32_t above = breaks >> (i + 1);
            const int left = above ? 1 + __builtin_ctz(above) : end - 8 * lane - i, reach = min(q, LZ_WINDOW);
            b.start_mask |= (uint32_t)((q < LZ_WINDOW ? q & (q - 1) : q & (LZ_WINDOW - 1)) == 0) << i;
            b.match_mask |= (uint32_t)(q != 0) << i;
            lens |= (uint64_t)min(reach, left) << (8 * i);
            offs |= (uint64_t)reach << (8 * i);
        }
        b.lens_lo = (uint32_t)lens; b.lens_hi = (uint32_t)(lens >> 32);
        b.offs_lo = (uint32_t)offs; b.offs_hi = (uint32_t)(offs >> 32);
        wave_sync();                                    // hmask is the key area of the next block
        b.count();
        return LZ_GENERAL;
    }

    // ---- the reference's matcher (gpulz.cu:46-85) on the masks: a run starts at the next hit,
    // grows while the following positions hit at the same distance, and the window symbol after
    // a run is consumed by the comparison that ended it.
    // The lengths of the runs that start at any bit come first, all bits at once: bit j is alive after k steps
    // if positions p .. p+k-1 hit at it, and when it dies k goes into the bit's place of six words.  (Run by run,
    // with a read of the following masks for each, a block whose first 64 symbols are zero took 45 us.)
    uint64_t lens = 0, offs = 0;
    b.match_mask = 0;
#pragma unroll 1
    for (uint32_t todo = live; todo != 0; todo &= todo - 1) {
        const int i = __builtin_ctz(todo);
        const uint32_t room = (uint32_t)(LZ_SYMS - 8 * lane - i);       // symbols left in the block
        const uint32_t mask = hmask[i * LZ_PITCH + lane];
        uint32_t alive = mask, runs[6] = {0, 0, 0, 0, 0, 0}, room_mask = 0x7fffffffu;
#pragma unroll 1
        for (int k0 = 0; k0 < LZ_WINDOW; k0 += 8) {
            if (__ballot(alive != 0) == 0) break;
            uint32_t next[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int at = i + k0 + t + 1;
                next[t] = hmask[(at & 7) * LZ_PITCH + lane + (at >> 3)];
            }
            // k = k0 + t + 1: a run of k ends here, or (32 - j symbols from bit j on) with the window.  Seven of the eight k share
            // their upper three bits; the eighth has the next ones and no lower bits.
            uint32_t low = 0, last = 0;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const uint32_t on = alive & next[t] & (room_mask >> t), dead = alive & ~on;
#pragma unroll
                for (int q = 0; q < 3; ++q) if (((t + 1) >> q) & 1) runs[q] |= dead;
                if (t < 7) low |= dead; else last = dead;
                alive = on;
            }
            room_mask >>= 8;
            const uint32_t here = (uint32_t)k0 >> 3, then = here + 1u;
#pragma unroll
            for (int q = 0; q < 3; ++q)
                runs[3 + q] |= (low & (0u - ((here >> q) & 1u))) | (last & (0u - ((then >> q) & 1u)));
        }
        uint32_t longest = 0, with = mask;              // of all runs, whether the walk gets to them or not
#pragma unroll
        for (int q = 5; q >= 0; --q)
            if (with & runs[q]) { with &= runs[q]; longest |= 1u << q; }
        uint32_t len = 0, off = 0, j = 0;
        while (len < longest && j + len < (uint32_t)LZ_WINDOW) {         // (no longer run to come)
            const uint32_t rest = mask & (0xffffffffu << j);
            if (rest == 0) break;
            const uint32_t j0 = __builtin_ctz(rest);
            uint32_t r = 0;
#pragma unroll
            for (int q = 0; q < 6; ++q) r |= ((runs[q] >> j0) & 1u) << q;
            if (r > len) { len = r; off = LZ_WINDOW - j0; }
            if (r >= room) break;                       // the look-ahead reached the end of the block
            j = j0 + r + 1;
        }
        lens |= (uint64_t)len << (8 * i);
        offs |= (uint64_t)off << (8 * i);
        b.match_mask |= (uint32_t)(len != 0) << i;
    }
    b.lens_lo = (uint32_t)lens; b.lens_hi = (uint32_t)(lens >> 32);
    b.offs_lo = (uint32_t)offs; b.offs_hi = (uint32_t)(offs >> 32);
    wave_sync();                                        // hmask is the key area of the next block

    // ---- greedy parse: [cur, nxt) is a run of literals, nxt the next position with a match
    b.start_mask = 0;
    int cur = 0;
    while (cur < LZ_SYMS) {
        const int rel = cur - 8 * lane;
        const uint32_t mm = rel >= 8 ? 0u : (rel <= 0 ? b.match_mask : (b.match_mask & (0xffu << rel)));
        const uint64_t bal = __ballot(mm != 0);
        int nxt = LZ_SYMS, step = 0;
        if (bal != 0) {
            const int owner = __builtin_ctzll(bal);
            const uint32_t m = __builtin_amdgcn_readlane(mm, owner);
            const int bit = __builtin_ctz(m);
            nxt = 8 * owner + bit;
            const uint32_t lo = __builtin_amdgcn_readlane(b.lens_lo, owner);
            const uint32_t hi = __builtin_amdgcn_readlane(b.lens_hi, owner);
            step = (int)(((bit < 4 ? lo : hi) >> (8 * (bit & 3))) & 0xffu);
        }
        // the literals and, when there is one, the match token at nxt all start a token
        const int last = bal != 0 ? nxt + 1 : nxt;
        const int lo_b = min(max(cur - 8 * lane, 0), 8);
        const int hi_b = min(max(last - 8 * lane, 0), 8);
        b.start_mask |= ((1u << hi_b) - 1u) & ~((1u << lo_b) - 1u);
        cur = nxt + step;                              // step >= 1 whenever nxt < 512
    }

    b.count();
    return LZ_GENERAL;
}

// ---- launch 1: sizes and class of every block.  WAVES: blocks of a work-group, which stays until the last of them is through.  Two where there are
// work-groups enough, eight otherwise (us to compress, 8 and 2: 32768 x 1024, 30 % empty 98.9, 93.4; 65536 x 1000 247, 223; 16384 x 512 34.6, 36.6;
// 8192 x 1024, none empty, 35.9, 37.1)
template <int WAVES>
__global__ __launch_bounds__(WAVES * WAVE) void lz_sizes_kernel(
    const uint32_t *__restrict__ in, int64_t nsym, int64_t blocks, int32_t *__restrict__ flag_off,
    int32_t *__restrict__ data_off, uint8_t *__restrict__ cls, uint32_t *__restrict__ sizes, uint4 *__restrict__ tokens, uint32_t *__restrict__ cleared)
{
    __shared__ __attribute__((aligned(16))) uint32_t keys[WAVES][LZ_WINDOW + LZ_SYMS];
    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int64_t block = (int64_t)blockIdx.x * WAVES + wave;
    if (block >= blocks) return;                       // no work-group barrier below
    uint32_t raw[8];
    lz_load(in, nsym, block, lane, raw);
    // (a buffer to be cleared along with it: the vector ALUs bound this launch, memory has time; 134 MB of it: a codec pass 163.5 us with a fill
    // of its own, 153.3)
    if (cleared) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t at = block * LZ_SYMS + (h * WAVE + lane) * 4;
            if (at + 4 <= nsym) __builtin_nontemporal_store(pm_u32x4{0u, 0u, 0u, 0u}, reinterpret_cast<pm_u32x4 *>(cleared + at));
            else for (int64_t i = at; i < nsym; ++i) cleared[i] = 0u;
        }
    }
    LzBlock b;
    const int c = lz_analyse(raw, keys[wave], lane, b);
    if (c == LZ_GENERAL) tokens[block * WAVE + lane] = b.tokens();
    if (lane == 0) {
        cls[block] = (uint8_t)c;
        if (sizes) {
            sizes[block] = b.flag_bytes | b.data_bytes << 16;
        } else {
            flag_off[block] = (int32_t)b.flag_bytes;
            data_off[block] = (int32_t)b.data_bytes;
            if (block == blocks - 1) { flag_off[blocks] = 0; data_off[blocks] = 0; }
        }
    }
}

// ---- launch 2: both tables, in place: exclusive sums inside chunks of 8192 entries, chunk totals
__global__ __launch_bounds__(256) void lz_scan_chunks_kernel(int32_t *__restrict__ flag_off,
                                                            int32_t *__restrict__ data_off, int64_t entries,
                                                            uint32_t *__restrict__ totals)
{
    __shared__ uint32_t wave_tot[4];
    constexpr int PER = LZ_SCAN_CHUNK / 256;            // 32 entries per thread, contiguous
    const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
    const int64_t e0 = (int64_t)blockIdx.x * LZ_SCAN_CHUNK + (int64_t)threadIdx.x * PER;
    const bool whole = e0 + PER <= entries;
    for (int a = 0; a < 2; ++a) {
        int32_t *t = a ? data_off : flag_off;
        uint32_t v[PER];
        if (whole) {
#pragma unroll
            for (int q = 0; q < PER / 4; ++q) {
                const int4 w = *reinterpret_cast<const int4 *>(t + e0 + 4 * q);
                v[4 * q] = (uint32_t)w.x; v[4 * q + 1] = (uint32_t)w.y; v[4 * q + 2] = (uint32_t)w.z; v[4 * q + 3] = (uint32_t)w.w;
            }
        } else {
#pragma unroll
            for (int q = 0; q < PER; ++q) v[q] = e0 + q < entries ? (uint32_t)t[e0 + q] : 0u;
        }
        uint32_t sum = 0;
#pragma unroll
        for (int q = 0; q < PER; ++q) sum += v[q];
        uint32_t total;
        uint32_t run = wave_exclusive_sum(sum, total);
        __syncthreads();                                // the totals of the other table have been read
        if (lane == 0) wave_tot[wave] = total;
        __syncthreads();
        for (int w = 0; w < wave; ++w) run += wave_tot[w];
#pragma unroll
        for (int q = 0; q < PER; ++q) { const uint32_t x = v[q]; v[q] = run; run += x; }
        if (whole) {
#pragma unroll
            for (int q = 0; q < PER / 4; ++q)
                *reinterpret_cast<int4 *>(t + e0 + 4 * q) =
                    make_int4((int)v[4 * q], (int)v[4 * q + 1], (int)v[4 * q + 2], (int)v[4 * q + 3]);
        } else {
#pragma unroll
            for (int q = 0; q < PER; ++q)
                if (e0 + q < entries) t[e0 + q] = (int32_t)v[q];
        }
        if (threadIdx.x == 255) totals[2 * blockIdx.x + a] = run;   // the last thread ends with the chunk's sum
    }
}

// the sums of the first n chunks' totals: flags, data
__device__ __forceinline__ uint2 lz_chunks_before(const uint32_t *__restrict__ totals, int n)
{
    uint32_t f = 0, d = 0;
    for (int c = lane_id(); c < n; c += WAVE) { f += totals[2 * c]; d += totals[2 * c + 1]; }
    auto sum = [](uint32_t a, uint32_t b) { return a + b; };
    return make_uint2((uint32_t)wave_allreduce((int)f, sum), (uint32_t)wave_allreduce((int)d, sum));
}

// zero flags[flag_total ..) and data[data_total ..): 16 bytes per lane and step, neighbouring lanes at
// neighbouring addresses (the piece the used part ends in byte by byte)
__device__ __forceinline__ void lz_clear_slack(int64_t tid, int64_t nthreads, int32_t flag_total, int32_t data_total,
                                               int64_t blocks, uint8_t *__restrict__ flags, uint8_t *__restrict__ data)
{
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        uint8_t *buf = a ? data : flags;
        const int64_t size = a ? blocks * LZ_BLOCK_BYTES : blocks * (LZ_SYMS / 8);     // multiples of 64
        const int64_t used = min(max((int64_t)(a ? data_total : flag_total), (int64_t)0), size);
        for (int64_t lo = (used / 16 + tid) * 16; lo < size; lo += nthreads * 16) {
            if (lo >= used) {
                *reinterpret_cast<uint4 *>(buf + lo) = make_uint4(0, 0, 0, 0);
            } else {
                for (int64_t q = used; q < lo + 16; ++q) buf[q] = 0;
            }
        }
    }
}

// the sums of the first n blocks' sizes and, in wave w, of w more: flags, data.  All waves of the work-group call it; n <= LZ_SUMMED
__device__ __forceinline__ uint2 lz_sizes_before(const uint32_t *__restrict__ sizes, int n, int more, int64_t blocks, uint32_t (*partial)[2])
{
    const int wave = (int)(threadIdx.x >> 6), lane = lane_id();
    const uint32_t own = sizes[min((int64_t)n + lane, blocks - 1)];
    uint32_t f = 0, d = 0;
    for (int i0 = threadIdx.x; i0 - (int)threadIdx.x < n; i0 += 4 * LZ_WAVES * WAVE) {
        uint32_t v[4];                                  // (straight-line loads at addresses that are there)
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = sizes[min(i0 + q * LZ_WAVES * WAVE, n - 1)];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t x = i0 + q * LZ_WAVES * WAVE < n ? v[q] : 0u;
            f += x & 0xffffu;
            d += x >> 16;
        }
    }
    auto sum = [](uint32_t a, uint32_t b) { return a + b; };
    f = (uint32_t)wave_allreduce((int)f, sum);
    d = (uint32_t)wave_allreduce((int)d, sum);
    if (lane == 0) { partial[wave][0] = f; partial[wave][1] = d; }
    __syncthreads();
    f = d = 0;
    if (lane < LZ_WAVES) { f = partial[lane][0]; d = partial[lane][1]; }
    if (lane < more) { f += own & 0xffffu; d += own >> 16; }
    return make_uint2((uint32_t)wave_allreduce((int)f, sum), (uint32_t)wave_allreduce((int)d, sum));
}

struct __attribute__((aligned(16))) LzPlaceShared {
    uint16_t stage[LZ_WAVES][LZ_BLOCK_BYTES / 2];   // token bytes of the block
    uint32_t flagw[LZ_WAVES][16];                   // flag bits of the block
};

// ---- the last launch: every block to its final place, and zeros behind the last.  SUMMED: by the blocks' sizes, without a scan before
template <bool SUMMED>
__global__ __launch_bounds__(LZ_WAVES * WAVE) void lz_place_kernel(
    const uint32_t *__restrict__ in, int64_t nsym, int64_t blocks, int32_t *__restrict__ flag_off,
    int32_t *__restrict__ data_off, const uint8_t *__restrict__ cls, const uint32_t *__restrict__ totals, int chunks, const uint32_t *__restrict__ sizes,
    const uint4 *__restrict__ tokens, uint8_t *__restrict__ flags, uint8_t *__restrict__ data)
{
    __shared__ LzPlaceShared sh;
    __shared__ uint32_t partial[LZ_WAVES][2];
    // the work-groups behind the blocks' clear what lies beyond the totals
    const int64_t groups = (blocks + LZ_WAVES - 1) / LZ_WAVES;
    if (blockIdx.x >= groups) {
        const uint2 all = SUMMED ? lz_sizes_before(sizes, (int)blocks, 0, blocks, partial) : lz_chunks_before(totals, chunks);
        lz_clear_slack(((int64_t)blockIdx.x - groups) * LZ_WAVES * WAVE + threadIdx.x, ((int64_t)gridDim.x - groups) * LZ_WAVES * WAVE,
                       (int32_t)all.x, (int32_t)all.y, blocks, flags, data);
        return;
    }
    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int64_t block = (int64_t)blockIdx.x * LZ_WAVES + wave;
    if (!SUMMED && block >= blocks) return;            // no work-group barrier below

    uint32_t raw[8];
    lz_load(in, nsym, block, lane, raw);
    uint2 before;
    if (SUMMED) {
        before = lz_sizes_before(sizes, (int)blockIdx.x * LZ_WAVES, wave, blocks, partial);
        if (block >= blocks) return;                   // no work-group barrier below
    } else {
        before = lz_chunks_before(totals, (int)(block / LZ_SCAN_CHUNK));
    }
    const uint32_t fbase = (SUMMED ? 0u : (uint32_t)flag_off[block]) + before.x;
    const uint32_t dbase = (SUMMED ? 0u : (uint32_t)data_off[block]) + before.y;
    int c = cls[block];
    c = __builtin_amdgcn_readfirstlane(c);
    // never let a wrong table move a write out of the buffers
    const uint32_t fb = min(fbase, (uint32_t)(block * (LZ_SYMS / 8)));
    const uint32_t db = min(dbase, (uint32_t)(block * LZ_BLOCK_BYTES)) & ~1u;
    uint2 all = make_uint2(0u, 0u);
    if (block == blocks - 1) {
        if (SUMMED) { const uint32_t own = sizes[block]; all = make_uint2(fbase + (own & 0xffffu), dbase + (own >> 16)); }
        else all = lz_chunks_before(totals, chunks);
    }
    if (lane == 0) {
        flag_off[block] = (int32_t)fbase;
        data_off[block] = (int32_t)dbase;
        if (block == blocks - 1) {                     // the totals sit in the entry after the last block
            flag_off[blocks] = (int32_t)all.x;
            data_off[blocks] = (int32_t)all.y;
        }
    }
    uint8_t *dst = data + db;
    uint16_t *stage = sh.stage[wave];
    uint32_t *flagw = sh.flagw[wave];
    uint32_t flag_bytes, data_bytes;

    if (c == LZ_STORED) {                              // 512 literals: the block itself, at an even address
        flags[(size_t)fb + lane] = 0;
        lz_u32x4_a2 *to = reinterpret_cast<lz_u32x4_a2 *>(dst);
        __builtin_nontemporal_store(pm_u32x4{raw[0], raw[1], raw[2], raw[3]}, to + 2 * lane);
        __builtin_nontemporal_store(pm_u32x4{raw[4], raw[5], raw[6], raw[7]}, to + 2 * lane + 1);
        return;
    } else if (c == LZ_CONSTANT) {
        flag_bytes = 3;
        data_bytes = 44;
        const uint32_t sym0 = __builtin_amdgcn_readfirstlane(raw[0]);
        if (lane < 22) {
            const uint32_t n = lane < 7 ? 1u << (lane - 2) : 32u;          // lanes 2..21: the 20 matches
            stage[lane] = (uint16_t)(lane == 0 ? sym0 : lane == 1 ? sym0 >> 16 : n | (n << 8));
        }
        if (lane == 0) flagw[0] = 0x001ffffeu;
    } else {
        const uint4 packed = tokens[block * WAVE + lane];
        const uint32_t words[4] = {packed.x, packed.y, packed.z, packed.w};
        auto token = [&](int i) { return words[i >> 1] >> (16 * (i & 1)); };
        LzBlock b;
        b.start_mask = b.match_mask = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            b.start_mask |= ((token(i) >> 15) & 1u) << i;
            b.match_mask |= ((token(i) >> 14) & 1u) << i;
        }
        b.count();
        flag_bytes = b.flag_bytes;
        data_bytes = b.data_bytes;
        if (lane < 16) flagw[lane] = 0;
        wave_sync();
        uint32_t bits = 0, nb = 0, at = b.byte_base >> 1;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if ((b.start_mask >> i) & 1) {
                if ((b.match_mask >> i) & 1) {
                    stage[at] = (uint16_t)(((token(i) & 0x1fu) + 1u) | ((((token(i) >> 5) & 0x1fu) + 1u) << 8));
                    at += 1;
                    bits |= 1u << nb;
                } else {
                    stage[at] = (uint16_t)raw[i];
                    stage[at + 1] = (uint16_t)(raw[i] >> 16);
                    at += 2;
                }
                ++nb;
            }
        }
        if (bits) {
            const uint64_t wide = (uint64_t)bits << (b.tok_base & 31u);
            atomicOr(&flagw[b.tok_base >> 5], (uint32_t)wide);
            if ((uint32_t)(wide >> 32)) atomicOr(&flagw[(b.tok_base >> 5) + 1], (uint32_t)(wide >> 32));
        }
    }
    wave_sync();
    if ((uint32_t)lane < flag_bytes)
        flags[(size_t)fb + lane] = (uint8_t)(flagw[lane >> 2] >> (8 * (lane & 3)));

    // token bytes: the offset is even; 2 bytes up to a 4-byte boundary, whole words, 2 bytes at the end
    const uint32_t head = (reinterpret_cast<uintptr_t>(dst) & 2u) ? 2u : 0u;
    if (head && lane == 0) *reinterpret_cast<uint16_t *>(dst) = stage[0];
    const uint32_t words = (data_bytes - head) >> 2;
    uint32_t *dw = reinterpret_cast<uint32_t *>(dst + head);
    for (uint32_t k = lane; k < words; k += WAVE) {
        const uint32_t h = (head >> 1) + 2 * k;
        stream_store(dw + k, (uint32_t)stage[h] | ((uint32_t)stage[h + 1] << 16));
    }
    if (((data_bytes - head) & 2u) && lane == 0)
        *reinterpret_cast<uint16_t *>(dst + data_bytes - 2) = stage[data_bytes / 2 - 1];
}

constexpr int LZ_DEC_WAVES = 2;          // a work-group's waves wait for its slowest: 65536 x 1000, 30 % empty, 1, 2, 4, 8 waves 74, 77, 84, 109 us

struct LzDecodeShared {
    uint32_t bytes[LZ_DEC_WAVES][LZ_BLOCK_BYTES / 4 + 1];  // token bytes of the block (one spare word)
    uint32_t out[LZ_DEC_WAVES][LZ_SYMS];
};

__device__ __forceinline__ uint32_t lds_u16(const uint32_t *words, uint32_t byte_at)   // byte_at even
{
    return (words[byte_at >> 2] >> (8 * (byte_at & 2u))) & 0xffffu;
}

// A block with matches (or at an odd address): tokens are laid out with two wave scans, literals
// land in parallel, matches follow in token order.  bytes / sym: LDS of the wavefront.
__device__ __forceinline__ void lz_decode_block(uint32_t *__restrict__ out, int64_t nsym, int64_t block, int lane,
                                                uint32_t fb, uint32_t nflag, int64_t d0, uint32_t nbytes,
                                                const uint8_t *__restrict__ data, uint32_t *bytes, uint32_t *sym)
{
    const int64_t s0 = block * LZ_SYMS + 8 * lane;
    // ---- stage the token bytes (source is 2-byte aligned), clear the output block
    {
        const uint8_t *src = data + d0;
        const uint32_t head = (reinterpret_cast<uintptr_t>(src) & 2u) ? 2u : 0u;    // bytes before a word boundary
        // word k of the staged block = source bytes 4k .. 4k+3
        for (uint32_t k = lane; k < LZ_BLOCK_BYTES / 4 + 1; k += WAVE) {
            uint32_t v = 0;
            if (4 * k < nbytes) {
                if (head == 0) {
                    // may run 2 bytes past nbytes; never past the buffer, whose size is a multiple of 4
                    v = *reinterpret_cast<const uint32_t *>(src + 4 * k);
                } else {
                    const uint32_t lo = *reinterpret_cast<const uint16_t *>(src + 4 * k);
                    const uint32_t hi = 4 * k + 2 < nbytes ? *reinterpret_cast<const uint16_t *>(src + 4 * k + 2) : 0u;
                    v = lo | (hi << 16);
                }
            }
            bytes[k] = v;
        }
        for (uint32_t k = lane; k < LZ_SYMS; k += WAVE) sym[k] = 0;
    }
    wave_sync();

    // ---- where each token's bytes and symbols start
    const uint32_t ntok_lane = (uint32_t)lane < nflag ? 8u : 0u;
    const uint32_t nm = __popc(fb);
    uint32_t total;
    uint32_t at = wave_exclusive_sum(4u * ntok_lane - 2u * nm, total);    // byte offset of the lane's first token
    uint32_t tok[8];                                   // match: pos | len << 10 | off << 18 | 1 << 31
    uint32_t nsyms = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        uint32_t t = 0;
        if ((uint32_t)lane < nflag) {
            if ((fb >> i) & 1) {
                const uint32_t lo = at < nbytes ? lds_u16(bytes, at) : 0u;
                t = ((lo & 0xffu) << 10) | ((lo >> 8) << 18) | (1u << 31);
                nsyms += lo & 0xffu;
                at += 2;
            } else {
                t = at << 10;                          // literal: remember where its bytes are
                nsyms += 1;
                at += 4;
            }
        }
        tok[i] = t;
    }
    uint32_t pos = wave_exclusive_sum(nsyms, total);
    uint32_t has_match = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if ((uint32_t)lane < nflag && pos < (uint32_t)LZ_SYMS) {
            if (tok[i] >> 31) {
                const uint32_t len = (tok[i] >> 10) & 0xffu, off = (tok[i] >> 18) & 0xffu;
                // a match of this coder lies inside the block and copies from before its start
                if (len != 0 && off >= len && off <= pos && pos + len <= (uint32_t)LZ_SYMS) {
                    tok[i] |= pos;
                    has_match |= 1u << i;
                }
                pos += len;
            } else {
                const uint32_t where = tok[i] >> 10;
                if (where + 4 <= nbytes)
                    sym[pos] = lds_u16(bytes, where) | (lds_u16(bytes, where + 2) << 16);
                pos += 1;
            }
        }
    }
    wave_sync();

    // ---- matches in token order: each copies symbols that are complete by then
    uint64_t pending = __ballot(has_match != 0);
    while (pending) {
        const int owner = __builtin_ctzll(pending);
        pending &= pending - 1;
        const uint32_t which = __builtin_amdgcn_readlane(has_match, owner);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (!((which >> i) & 1)) continue;
            const uint32_t t = __builtin_amdgcn_readlane(tok[i], owner);
            const uint32_t p = t & 0x3ffu, len = (t >> 10) & 0xffu, off = (t >> 18) & 0xffu;
            if ((uint32_t)lane < len) sym[p + lane] = sym[p - off + lane];
            wave_sync();
        }
    }

    // ---- write the block
    const uint4 a = *reinterpret_cast<const uint4 *>(sym + 8 * lane);
    const uint4 b = *reinterpret_cast<const uint4 *>(sym + 8 * lane + 4);
    if (s0 + 8 <= nsym) {
        stream_store(reinterpret_cast<uint4 *>(out + s0), a);
        stream_store(reinterpret_cast<uint4 *>(out + s0 + 4), b);
    } else {
        const uint32_t v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (s0 + i < nsym) out[s0 + i] = v[i];
    }
}

// A wave a block.  (Two and four blocks a wave with their loads in flight together wait for each other where blocks have matches: us of 1, 2 and 4,
// 134 MB with 30 % empty slots 37.5, 38.5, 39.8; 10 MB, rows of 640, 9.1, 13.4, 18.7; 400 rows of 300, half of them empty, 7.8, 13.0, 23.2.)
__global__ __launch_bounds__(LZ_DEC_WAVES * WAVE) void lz_decompress_kernel(
    uint32_t *__restrict__ out, int64_t nsym, int64_t blocks, const int32_t *__restrict__ flag_off,
    const int32_t *__restrict__ data_off, const uint8_t *__restrict__ flags,
    const uint8_t *__restrict__ data)
{
    __shared__ LzDecodeShared sh;
    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int64_t block = (int64_t)blockIdx.x * LZ_DEC_WAVES + wave;
    if (block >= blocks) return;                       // no work-group barrier below

    // All loads up to the first branch are unconditional, at clamped addresses: a load under a branch would make
    // every later wait drain the whole queue.
    // offsets of a stream of this coder ascend and stay inside the buffers; clamp all the same
    const int64_t fcap = blocks * (LZ_SYMS / 8), dcap = blocks * LZ_BLOCK_BYTES;
    const int64_t f0 = min(max((int64_t)flag_off[block], (int64_t)0), fcap), d0 = min(max((int64_t)data_off[block], (int64_t)0), dcap) & ~(int64_t)1;
    const int64_t f1 = min(max((int64_t)flag_off[block + 1], f0), min(f0 + LZ_SYMS / 8, fcap));
    const int64_t d1 = min(max((int64_t)data_off[block + 1], d0), min(d0 + LZ_BLOCK_BYTES, dcap));
    const uint32_t nflag = (uint32_t)(f1 - f0), nbytes = (uint32_t)(d1 - d0);
    // a stored block (512 literals) is its own bytes: fetch them before the flags are known
    const bool whole = block * LZ_SYMS + LZ_SYMS <= nsym, direct = nflag == LZ_SYMS / 8 && nbytes == LZ_BLOCK_BYTES && whole;
    const uint32_t fb = flags[min(f0 + lane, fcap - 1)];                   // lane l: tokens 8l .. 8l+7
    const lz_u32x4_a2 *src = reinterpret_cast<const lz_u32x4_a2 *>(data + (direct ? d0 : 0));
    const pm_u32x4 va = src[lane], vb = src[lane + WAVE];                  // 1 KB per instruction
    pm_u32x4 *dst = reinterpret_cast<pm_u32x4 *>(out + block * LZ_SYMS);
    if (direct && __ballot((uint32_t)lane < nflag && fb != 0) == 0) {
        __builtin_nontemporal_store(va, dst + lane);
        __builtin_nontemporal_store(vb, dst + lane + WAVE);
        return;
    }
    // Blocks of one repeated value (empty capacity slots): this coder's 44 bytes for it -- the value, (1,1) (2,2) (4,4) (8,8)
    // (16,16) and (32,32) to the end -- are recognised as a whole and not walked match by match.  (134 MB with 30 % of its slots
    // empty: 70 us when they were walked.)
    if (nflag == 3 && nbytes == 44 && whole) {
        const uint32_t token = *reinterpret_cast<const uint16_t *>(data + min(d0 + 2 * min(lane, 21), dcap - 2));
        const uint32_t n = lane < 7 ? 1u << max(lane - 2, 0) : 32u, flag = lane == 0 ? 0xfeu : lane == 1 ? 0xffu : 0x1fu;
        if (__ballot((lane >= 2 && lane < 22 && token != (n | (n << 8))) || (lane < 3 && fb != flag)) == 0) {
            const uint32_t v = __builtin_amdgcn_readlane(token, 0) | (__builtin_amdgcn_readlane(token, 1) << 16);
            __builtin_nontemporal_store(pm_u32x4{v, v, v, v}, dst + lane);
            __builtin_nontemporal_store(pm_u32x4{v, v, v, v}, dst + lane + WAVE);
            return;
        }
    }
    lz_decode_block(out, nsym, block, lane, (uint32_t)lane < nflag ? fb : 0u, nflag, d0, nbytes, data, sh.bytes[wave], sh.out[wave]);
}

int lz_check(const char *who, int64_t nbytes)
{
    PM_REQUIRE(nbytes >= 0 && nbytes % 4 == 0, "%s: nbytes must be a non-negative multiple of 4 (got %lld)", who,
               (long long)nbytes);
    PM_REQUIRE(nbytes + LZ_BLOCK_BYTES <= (1ll << 31), "%s: nbytes too large for int32 offsets (%lld)", who,
               (long long)nbytes);
    return 0;
}

} // namespace
} // namespace pm

using namespace pm;

extern "C" int64_t planmoe_lz_blocks(int64_t nbytes)
{
    return nbytes <= 0 ? 0 : (nbytes + LZ_BLOCK_BYTES - 1) / LZ_BLOCK_BYTES;
}

// workspace: class byte per block | chunk totals | sizes of LZ_SUMMED blocks at most (unused by more, but counted: what serves an input serves every shorter
// one) | tokens of the blocks with matches, two bytes a position
static size_t lz_class_bytes(int64_t blocks) { return round_up((size_t)blocks, 256); }
static size_t lz_sizes_at(int64_t blocks) { return lz_class_bytes(blocks) + 2 * LZ_MAX_CHUNKS * sizeof(uint32_t); }
static size_t lz_tokens_at(int64_t blocks) { return lz_sizes_at(blocks) + round_up((size_t)min(blocks, (int64_t)LZ_SUMMED) * 4, 256); }

extern "C" size_t planmoe_lz_workspace_bytes(int64_t nbytes)
{
    const int64_t blocks = planmoe_lz_blocks(nbytes);
    return lz_tokens_at(blocks) + 16 + (size_t)blocks * LZ_SYMS * 2;       // (the tokens begin at the next 16 bytes)
}

static int lz_compress_and_clear(const char *who, const void *input, int64_t nbytes, int32_t *flag_offsets, int32_t *data_offsets, uint8_t *flags,
                                 uint8_t *data, void *workspace, size_t workspace_bytes, void *cleared, void *stream)
{
    if (lz_check(who, nbytes)) return 1;
    PM_REQUIRE(flag_offsets && data_offsets, "%s: offset tables must not be NULL", who);
    hipStream_t st = (hipStream_t)stream;
    const int64_t blocks = planmoe_lz_blocks(nbytes);
    if (blocks == 0) {
        fill_u32((uint32_t *)flag_offsets, 1, 0u, st);
        fill_u32((uint32_t *)data_offsets, 1, 0u, st);
        PM_LAUNCH_CHECK(who);
        return 0;
    }
    PM_REQUIRE(input && flags && data, "%s: NULL argument", who);
    PM_REQUIRE(aligned16(input) && aligned16(flags) && aligned16(data) && aligned16(flag_offsets) &&
               aligned16(data_offsets),
               "%s: input, flags, data and the offset tables must be 16-byte aligned", who);
    PM_REQUIRE(workspace && workspace_bytes >= planmoe_lz_workspace_bytes(nbytes) &&
               (reinterpret_cast<uintptr_t>(workspace) & 3u) == 0,
               "%s: workspace too small or not 4-byte aligned", who);
    uint8_t *cls = (uint8_t *)workspace;
    uint32_t *totals = (uint32_t *)(cls + lz_class_bytes(blocks));
    const bool summed = blocks <= LZ_SUMMED;
    uint32_t *sizes = summed ? (uint32_t *)(cls + lz_sizes_at(blocks)) : nullptr;
    uint4 *tokens = (uint4 *)(((uintptr_t)workspace + lz_tokens_at(blocks) + 15) / 16 * 16);
    const int64_t groups = (blocks + LZ_WAVES - 1) / LZ_WAVES;
    const int64_t entries = blocks + 1;
    const int chunks = (int)((entries + LZ_SCAN_CHUNK - 1) / LZ_SCAN_CHUNK);      // <= 128 below 2^31 bytes
    const int64_t waves = blocks > 2 * LZ_SUMMED ? 2 : LZ_WAVES;
    const auto classify = waves == 2 ? lz_sizes_kernel<2> : lz_sizes_kernel<LZ_WAVES>;
    classify<<<(unsigned)((blocks + waves - 1) / waves), waves * WAVE, 0, st>>>((const uint32_t *)input, nbytes / 4, blocks,
                                                                flag_offsets, data_offsets, cls, sizes, tokens, (uint32_t *)cleared);
    if (!summed) lz_scan_chunks_kernel<<<chunks, 256, 0, st>>>(flag_offsets, data_offsets, entries, totals);
    const int64_t slack_chunks = (blocks * LZ_BLOCK_BYTES / 16 + 255) / 256;          // enough for all of data
    const int64_t clear_groups = min((slack_chunks + 1) / 2, (int64_t)(chunks > 1 ? 2048 : 256));
    const auto place = summed ? lz_place_kernel<true> : lz_place_kernel<false>;
    place<<<(unsigned)(groups + clear_groups), LZ_WAVES * WAVE, 0, st>>>((const uint32_t *)input, nbytes / 4, blocks, flag_offsets, data_offsets, cls, totals, chunks,
                                                                       sizes, tokens, flags, data);
    PM_LAUNCH_CHECK(who);
    return 0;
}

extern "C" int planmoe_lz_compress(const void *input, int64_t nbytes, int32_t *flag_offsets,
                                   int32_t *data_offsets, uint8_t *flags, uint8_t *data, void *workspace,
                                   size_t workspace_bytes, void *stream)
{
    return lz_compress_and_clear("planmoe_lz_compress", input, nbytes, flag_offsets, data_offsets, flags, data, workspace, workspace_bytes, nullptr, stream);
}

extern "C" int planmoe_lz_compress_clearing(const void *input, int64_t nbytes, int32_t *flag_offsets,
                                            int32_t *data_offsets, uint8_t *flags, uint8_t *data, void *cleared,
                                            void *workspace, size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_lz_compress_clearing";
    PM_REQUIRE((cleared && aligned16(cleared)) || nbytes == 0, "%s: the buffer to clear is NULL or not 16-byte aligned", who);
    return lz_compress_and_clear(who, input, nbytes, flag_offsets, data_offsets, flags, data, workspace, workspace_bytes, cleared, stream);
}

extern "C" int planmoe_lz_decompress(void *output, int64_t nbytes, const int32_t *flag_offsets,
                                     const int32_t *data_offsets, const uint8_t *flags, const uint8_t *data,
                                     void *stream)
{
    if (lz_check("planmoe_lz_decompress", nbytes)) return 1;
    const int64_t blocks = planmoe_lz_blocks(nbytes);
    if (blocks == 0) return 0;
    PM_REQUIRE(output && flag_offsets && data_offsets && flags && data, "planmoe_lz_decompress: NULL argument");
    PM_REQUIRE(aligned16(output) && (reinterpret_cast<uintptr_t>(data) & 3u) == 0,
               "planmoe_lz_decompress: output must be 16-byte and data 4-byte aligned");
    const int64_t groups = (blocks + LZ_DEC_WAVES - 1) / LZ_DEC_WAVES;
    lz_decompress_kernel<<<(unsigned)groups, LZ_DEC_WAVES * WAVE, 0, (hipStream_t)stream>>>(
        (uint32_t *)output, nbytes / 4, blocks, flag_offsets, data_offsets, flags, data);
    PM_LAUNCH_CHECK("planmoe_lz_decompress");
    return 0;
}
