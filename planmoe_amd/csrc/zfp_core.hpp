// The coder and the decoder of a zfp block (4 or 4 x 4 values) in registers.
#pragma once
#include "common.hpp"
#include <cmath>

namespace pm {

// The words of a block's bit stream are parked in LDS while the block is coded (word i of thread
// t at lds[i * 256 + t]): a register array would need a select per word on every flush, since
// the word index differs from lane to lane.
template <int NW>
struct BitWriter {
    uint32_t *slot;
    uint64_t acc;
    int fill;
    __device__ __forceinline__ void init(uint32_t *lds)
    {
        slot = lds + threadIdx.x;
#pragma unroll
        for (int i = 0; i < NW; ++i) slot[i * 256] = 0u;
        acc = 0; fill = 0;
    }
    // append the low n (<= 32) bits of v; bits of v above n must be zero
    __device__ __forceinline__ void put(uint32_t v, int n)
    {
        acc |= (uint64_t)v << fill;
        fill += n;
        if (fill >= 32) { *slot = (uint32_t)acc; slot += 256; acc >>= 32; fill -= 32; }
    }
    __device__ __forceinline__ void finish() { if (fill > 0) *slot = (uint32_t)acc; }
    __device__ __forceinline__ void words(uint32_t *lds, uint32_t *w) const
    {
#pragma unroll
        for (int i = 0; i < NW; ++i) w[i] = lds[i * 256 + threadIdx.x];
    }
};

// The decoder looks at the stream by bit position: the block's words sit in LDS (NW words per
// thread and three zero words behind them: an odd stride) and a look is neighbouring words
// funnel-shifted, so there is no refill state to carry and no branch in the reader.  A bit plane
// takes one look of 64 bits (a plane never uses more than 48) and is then parsed in registers: the
// group tests of a 2-D block eight stream bits at a time by table (gt16_step), except the plane the
// block's budget ends in, which is walked bit by bit.
// Streams of one or two words stay in a register pair that is shifted as bits are consumed.
template <int NW>
struct BitReader {
    static constexpr int STRIDE = NW + 3;
    const uint32_t *words;      // this thread's NW + 3 words in LDS
    int pos;
    uint64_t small;             // NW <= 2: the whole stream in a register pair instead
    __device__ __forceinline__ void init(uint32_t *lds, const uint32_t *w)
    {
        pos = 0;
        if constexpr (NW <= 2) {
            small = w[0];
            if constexpr (NW == 2) small |= (uint64_t)w[1] << 32;
            words = nullptr;
        } else {
            uint32_t *mine = lds + threadIdx.x * STRIDE;
#pragma unroll
            for (int i = 0; i < NW; ++i) mine[i] = w[i];
            mine[NW] = 0u;
            mine[NW + 1] = 0u;
            mine[NW + 2] = 0u;
            words = mine;
            small = 0;
        }
    }
    // the next 32 bits of the stream (zeros past its end)
    __device__ __forceinline__ uint32_t peek() const
    {
        if constexpr (NW <= 2) {
            return (uint32_t)small;                 // skip() keeps the register pair shifted
        } else {
            const int i = pos >> 5;
            return __builtin_amdgcn_alignbit(words[i + 1], words[i], pos & 31);
        }
    }
    // the next 64 bits
    __device__ __forceinline__ uint64_t peek64() const
    {
        if constexpr (NW <= 2) {
            return small;
        } else {
            const int i = pos >> 5, sh = pos & 31;
            const uint32_t w0 = words[i], w1 = words[i + 1], w2 = words[i + 2];
            return (uint64_t)__builtin_amdgcn_alignbit(w1, w0, sh) | ((uint64_t)__builtin_amdgcn_alignbit(w2, w1, sh) << 32);
        }
    }
    __device__ __forceinline__ void skip(int n)      // n <= 32 (NW <= 2), any n otherwise
    {
        if constexpr (NW <= 2) small >>= n;
        else pos += n;
    }
    __device__ __forceinline__ uint32_t get(int n)   // n <= 31
    {
        const uint32_t v = peek() & ((1u << n) - 1u);
        skip(n);
        return v;
    }
};

__device__ __forceinline__ void fwd_lift(int32_t &x, int32_t &y, int32_t &z, int32_t &w)
{
    x += w; x >>= 1; w -= x;
    z += y; z >>= 1; y -= z;
    x += z; x >>= 1; z -= x;
    w += y; w >>= 1; y -= w;
    w += y >> 1; y -= w >> 1;
}

__device__ __forceinline__ void inv_lift(int32_t &x, int32_t &y, int32_t &z, int32_t &w)
{
    y += w >> 1; w -= y >> 1;
    y += w; w = (int32_t)((uint32_t)w << 1); w -= y;
    z += x; x = (int32_t)((uint32_t)x << 1); x -= z;
    y += z; z = (int32_t)((uint32_t)z << 1); z -= y;
    w += x; x = (int32_t)((uint32_t)x << 1); x -= w;
}

__device__ __forceinline__ uint32_t to_negabinary(int32_t v) { return ((uint32_t)v + 0xaaaaaaaau) ^ 0xaaaaaaaau; }
__device__ __forceinline__ int32_t from_negabinary(uint32_t v) { return (int32_t)((v ^ 0xaaaaaaaau) - 0xaaaaaaaau); }

// 16 x 16 bit matrix transpose.  w[j] holds row 2j in its low and row 2j+1 in its high half;
// afterwards bit i of row k is what bit k of row i was.  Used to turn the upper halves of the 16
// coefficients of a 2-D block into their 16 upper bit planes (and back) in about 100
// instructions instead of 32 per plane.
__device__ __forceinline__ void transpose16(uint32_t (&w)[8])
{
    auto swap_blocks = [](uint32_t &a, uint32_t &b, int s, uint32_t m) {
        const uint32_t t = ((a >> s) ^ b) & m;
        b ^= t; a ^= t << s;
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) swap_blocks(w[j], w[j + 4], 8, 0x00ff00ffu);
    swap_blocks(w[0], w[2], 4, 0x0f0f0f0fu); swap_blocks(w[1], w[3], 4, 0x0f0f0f0fu);
    swap_blocks(w[4], w[6], 4, 0x0f0f0f0fu); swap_blocks(w[5], w[7], 4, 0x0f0f0f0fu);
#pragma unroll
    for (int j = 0; j < 8; j += 2) swap_blocks(w[j], w[j + 1], 2, 0x33333333u);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t t = ((w[j] >> 15) ^ w[j]) & 0x0000aaaau;
        w[j] ^= t | (t << 15);
    }
}

// sequency order of the 4x4 coefficients (index into the i + 4j block layout)
__device__ constexpr int perm2(int i)
{
    constexpr int P[16] = {0, 1, 4, 5, 2, 8, 6, 9, 3, 12, 10, 7, 13, 11, 14, 15};
    return P[i];
}

// Group-test code of one bit plane without a data-dependent loop.
// For the not yet significant part r of a plane (bit p = value nsig + p) zfp emits, segment by
// segment, a test bit '1', the zeros below the next one bit and that one bit; i.e. the bits of r
// up to its highest one with a '1' put in front of bit 0 and of every bit that follows a one.
// The table holds that expansion for 8 bits of r at a time: entry [prev][byte] = code in the low
// 16 bits, its length (8 + prev + ones among the low 7 bits) above.  What follows the highest
// one (a single '0' test bit, or nothing at the block end) and the implicit last one are a
// matter of the total length, see encode_block.
__host__ __device__ constexpr uint32_t group_code_entry(int prev, int byte)
{
    uint32_t code = 0; int len = 0;
    for (int p = 0; p < 8; ++p) {
        const int bit = (byte >> p) & 1;
        if (prev) { code |= 1u << len; ++len; }
        code |= (uint32_t)bit << len; ++len;
        prev = bit;
    }
    return code | ((uint32_t)len << 16);
}
// all 256 threads of the work-group; tab has 512 entries
__device__ __forceinline__ void group_code_table(uint32_t *tab)
{
    tab[threadIdx.x] = group_code_entry(0, threadIdx.x);
    tab[256 + threadIdx.x] = group_code_entry(1, threadIdx.x);
    __syncthreads();
}
// the same where no work-group fills one
struct GroupCodeTable {
    uint32_t entry[512];
    constexpr GroupCodeTable() : entry()
    {
        for (int i = 0; i < 512; ++i) entry[i] = group_code_entry(i >> 8, i & 255);
    }
};
__constant__ const GroupCodeTable group_codes = GroupCodeTable();
__device__ __forceinline__ uint32_t low_bits(int n) { return (uint32_t)(((uint64_t)1 << n) - 1u); }   // n in 0..32

// N = values per block (4 or 16).  f is consumed; the block's maxbits = 32*NW bits land in bw.
template <int N, int NW>
__device__ __forceinline__ void encode_block(const float *f, BitWriter<NW> &bw, uint32_t *lds,
                                             const uint32_t *tab)
{
    bw.init(lds);
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) m = fmaxf(m, fabsf(f[i]));
    if (!(m > 0.f)) return;                       // all-zero block: '0' flag and zero padding
    // frexp exponent clamped at 1 - 127, i.e. exponent field - 126 (a denormal maximum reads 0)
    const int field = (int)((__float_as_uint(m) >> 23) & 0xffu);
    const int emax = field - 126;
    bw.put(2u * (uint32_t)(emax + 127) + 1u, 9);

    // block-floating-point cast: q = (int32)(f * 2^(30 - emax)), x86 conversion on overflow
    const int se = 30 - emax;
    const float s = se > 127 ? INFINITY : __uint_as_float((uint32_t)(se + 127) << 23);
    int32_t q[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float v = f[i] * s;
        // -2^31 itself converts to INT_MIN either way
        q[i] = fabsf(v) < 2147483648.0f ? (int32_t)v : (int32_t)0x80000000;
    }
    uint32_t u[N];
    if constexpr (N == 4) {
        fwd_lift(q[0], q[1], q[2], q[3]);
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = to_negabinary(q[i]);
    } else {
#pragma unroll
        for (int y = 0; y < 4; ++y) fwd_lift(q[4 * y], q[4 * y + 1], q[4 * y + 2], q[4 * y + 3]);
#pragma unroll
        for (int x = 0; x < 4; ++x) fwd_lift(q[x], q[x + 4], q[x + 8], q[x + 12]);
#pragma unroll
        for (int i = 0; i < 16; ++i) u[i] = to_negabinary(q[perm2(i)]);
    }

    // embedded coding: bit planes from the top, group-tested, until the budget is spent
    int bits = 32 * NW - 9;
    int nsig = 0;
    auto code_plane = [&](uint32_t x) __attribute__((always_inline)) {
        const int mm = min(nsig, bits);
        bits -= mm;
        bw.put(x & ((1u << mm) - 1u), mm);
        if (nsig < N && bits > 0) {
            const uint32_t r = x >> mm;                   // mm == nsig here
            // r == 0 runs through the same formulas: top = -1, no code bits, length 1 (the '0')
            const int top = 31 - __clz((int)r), ones = __builtin_popcount(r);
            const uint32_t e0 = tab[256 + (r & 0xffu)];
            uint32_t code = e0 & 0xffffu;
            if constexpr (N > 8) {
                const uint32_t e1 = tab[((r >> 7) & 1u) * 256 + (r >> 8)];
                code |= (e1 & 0xffffu) << (e0 >> 16);
            }
            // cut after the highest one bit (not emitted when it is the block's last value),
            // then one more '0' test bit unless the block ends there
            const int last = nsig + top == N - 1;
            const int lt = top + 1 + ones - last;
            const int len = lt + (nsig + top + 1 < N ? 1 : 0);
            const int emit = min(len, bits);
            code &= low_bits(min(lt, emit));
            bw.put(code, emit);
            bits -= emit;
            nsig += top + 1;
        }
    };
    if constexpr (N == 16) {
        // planes 31..16 by one bit transpose of the coefficients' upper halves
        uint32_t w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] = (u[2 * j] >> 16) | (u[2 * j + 1] & 0xffff0000u);
        transpose16(w);
#pragma unroll
        for (int k = 15; k >= 0; --k)
            if (bits > 0) code_plane((k & 1) ? w[k >> 1] >> 16 : w[k >> 1] & 0xffffu);
        for (int k = 15; k >= 0 && bits > 0; --k) {
            uint32_t x = 0;
#pragma unroll
            for (int i = 0; i < N; ++i) x |= ((u[i] >> k) & 1u) << i;
            code_plane(x);
        }
    } else {
        for (int k = 31; k >= 0 && bits > 0; --k) {
            uint32_t x = 0;
#pragma unroll
            for (int i = 0; i < N; ++i) x |= ((u[i] >> k) & 1u) << i;
            code_plane(x);
        }
    }
    bw.finish();
}

// ---- group tests of a 2-D block's bit plane, eight stream bits at a time
// The group-test bits of a plane are a walk with two states: a test bit is due (T), or the zeros of
// a run up to the next one bit are being read (R).  What eight stream bits do to that walk depends
// on the state and on how far away the block's last value is (its one is implied, and after it the
// plane ends without another test bit).  gt16_step works that out once per (state, distance, byte):
// bits 0..7 the one bits found (relative to the first value that was not significant), bits 8..11
// the values passed, bits 12..15 a code c: c <= 8 = the plane ended after c bits; 9 / 10 = all eight
// bits used and the walk goes on in state T / R.  The walk is zfp's own (decode_ints), minus the
// budget: a step that would use up the budget is not taken, see fast_plane16.
__host__ __device__ constexpr uint16_t gt16_step(int state, int r, uint32_t byte)
{
    const int last = r < 8 ? r : 99;            // the block's last value, if this step can reach it
    int n = 0, used = 0, st = state;
    uint32_t mask = 0;
    bool done = false;
    while (true) {
        if (st == 0) {
            if (n > last) { done = true; break; }
            if (used == 8) break;
            const uint32_t b = (byte >> used) & 1u; ++used;
            if (!b) { done = true; break; }
            st = 1;
        }
        bool out_of_bits = false;
        while (n != last) {
            if (used == 8) { out_of_bits = true; break; }
            const uint32_t b = (byte >> used) & 1u; ++used;
            if (b) break;
            ++n;
        }
        if (out_of_bits) break;
        mask |= 1u << n; ++n; st = 0;
        if (n > last) { done = true; break; }
    }
    const int c = done ? used : (st ? 10 : 9);
    return (uint16_t)(mask | ((uint32_t)n << 8) | ((uint32_t)c << 12));
}
constexpr int GT16_ENTRIES = 9 * 2 * 256;      // [min(15 - nsig, 8)][state][byte]
struct Gt16Table {
    uint16_t step[GT16_ENTRIES];
    constexpr Gt16Table() : step()
    {
        for (int i = 0; i < GT16_ENTRIES; ++i) step[i] = gt16_step((i >> 8) & 1, i >> 9, (uint32_t)i & 255u);
    }
};
__constant__ const Gt16Table gt16_table = Gt16Table();

// all 256 threads of the work-group copy the table into LDS (9 KB); a barrier follows
__device__ __forceinline__ void gt16_load(uint16_t *tab)
{
    const uint32_t *src = reinterpret_cast<const uint32_t *>(gt16_table.step);
    uint32_t *dst = reinterpret_cast<uint32_t *>(tab);
#pragma unroll
    for (int i = 0; i < GT16_ENTRIES / 2 / 256; ++i) dst[threadIdx.x + 256 * i] = src[threadIdx.x + 256 * i];
    __syncthreads();
}

// One bit plane of a 2-D block, bit by bit as zfp walks it: look = the next 64 stream bits (a plane
// never uses more than 48), bits = what is left of the block's budget, nsig = values significant so
// far.  nsig verbatim bits, then segment by segment the test bit and the zeros up to the next one
// bit (cut short by the budget or by the block's last value, whose one is implied).
__device__ __forceinline__ uint32_t slow_plane16(uint64_t look, int &bits, int &nsig)
{
    constexpr int N = 16;
    const int mm = min(nsig, bits);
    bits -= mm;
    uint32_t x = (uint32_t)look & ((1u << mm) - 1u);
    look >>= mm;
    while (nsig < N && bits > 0) {
        const uint32_t lo = (uint32_t)look;
        if (!(lo & 1u)) { --bits; break; }
        const int lim = min(N - 1 - nsig, bits - 1);
        const uint32_t win = (lo >> 1) & ((1u << lim) - 1u);
        const int z = win != 0u ? __builtin_ctz(win) : lim;       // zeros read
        const int used = 1 + (win != 0u ? z + 1 : lim);
        look >>= used; bits -= used; nsig += z;
        x |= 1u << nsig;
        ++nsig;
    }
    return x;
}

// The same plane by table, as long as the budget does not end inside it: false = it would (bits and
// nsig are then whatever the walk left them at: the caller keeps its own copies and has
// slow_plane16 do that plane, the block's last).  One exit and selects instead of branches: the
// lanes of a wave are at different points of their walks.
__device__ __forceinline__ bool fast_plane16(uint64_t look, int &bits, int &nsig, uint32_t &x, const uint16_t *tab)
{
    const int mm = min(nsig, bits);
    bits -= mm;
    x = (uint32_t)look & ((1u << mm) - 1u);
    look >>= mm;
    bool over = false, go = nsig < 16 && bits > 0;
    uint32_t st = 0u;                          // state * 256
    while (go) {
        const uint32_t r = (uint32_t)min(15 - nsig, 8);
        const uint32_t e = tab[(r << 9) | st | ((uint32_t)look & 255u)];
        const uint32_t c = e >> 12;
        const int used = (int)min(c, 8u);
        over = used >= bits;
        const int u = over ? 0 : used;
        x |= (over ? 0u : (e & 255u)) << nsig;
        nsig += over ? 0 : (int)((e >> 8) & 15u);
        look >>= u; bits -= u;
        st = (c & 1u) ? 0u : 256u;             // c = 9: state T, c = 10: state R (other values end the walk)
        go = !over && c >= 9u;
    }
    return !over;
}

// tab: the group-test table in LDS (gt16_load), used by 2-D blocks only
template <int N, int NW>
__device__ __forceinline__ void decode_block(BitReader<NW> &br, float *f, const uint16_t *tab = nullptr)
{
    if (!br.get(1)) {
#pragma unroll
        for (int i = 0; i < N; ++i) f[i] = 0.f;
        return;
    }
    const int emax = (int)br.get(8) - 127;
    uint32_t u[N];
#pragma unroll
    for (int i = 0; i < N; ++i) u[i] = 0u;
    int bits = 32 * NW - 9;
    int nsig = 0;
    auto read_plane = [&]() __attribute__((always_inline)) {
        if constexpr (N == 4) {
            const int mm = min(nsig, bits);
            bits -= mm;
            uint32_t x = br.get(mm);
            while (nsig < N && bits > 0) {
                // tiny blocks: test bit and run are read separately (measured faster here)
                --bits;
                if (!br.get(1)) break;
                const int lim = min(N - 1 - nsig, bits);
                const uint32_t win = br.peek() & ((1u << lim) - 1u);
                const int z = win != 0u ? __builtin_ctz(win) : lim;
                const int used = win != 0u ? z + 1 : lim;
                br.skip(used); bits -= used; nsig += z;
                x |= 1u << nsig;
                ++nsig;
            }
            return x;
        } else {
            // one look at the stream per plane
            const int before = bits;
            const uint32_t x = slow_plane16(br.peek64(), bits, nsig);
            br.skip(before - bits);
            return x;
        }
    };
    if constexpr (N == 16) {
        // planes 31..16 are collected as rows and transposed into the coefficients' upper halves
        uint32_t w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] = 0u;
        // by table, up to the plane the budget ends in: that one is set aside (every lane has one, each
        // at a plane of its own) and walked bit by bit afterwards, by all lanes at once
        int last_k = -1, last_bits = 0, last_nsig = 0;
        uint64_t last_look = 0;
#pragma unroll
        for (int k = 15; k >= 0; --k) {
            // (a branch of the whole wave; a lane whose budget is spent walks a plane of no bits)
            if (__builtin_amdgcn_ballot_w64(bits > 0) != 0) {
                const uint64_t look = br.peek64();
                const int before = bits, nsig0 = nsig;
                uint32_t x;
                const bool ok = fast_plane16(look, bits, nsig, x, tab);
                br.skip(ok ? before - bits : 0);
                w[k >> 1] |= ok ? x << (16 * (k & 1)) : 0u;
                last_k = ok ? last_k : k;
                last_look = ok ? last_look : look;
                last_bits = ok ? last_bits : before;
                last_nsig = ok ? last_nsig : nsig0;
                bits = ok ? bits : 0;
            }
        }
        if (last_k >= 0) {
            const uint32_t x = slow_plane16(last_look, last_bits, last_nsig) << (16 * (last_k & 1));
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] |= (last_k >> 1) == j ? x : 0u;
        }
        transpose16(w);
#pragma unroll
        for (int j = 0; j < 8; ++j) { u[2 * j] = w[j] << 16; u[2 * j + 1] = w[j] & 0xffff0000u; }
        for (int k = 15; k >= 0 && bits > 0; --k) {
            const uint32_t x = read_plane();
#pragma unroll
            for (int i = 0; i < N; ++i) u[i] |= ((x >> i) & 1u) << k;
        }
    } else {
        for (int k = 31; k >= 0 && bits > 0; --k) {
            const uint32_t x = read_plane();
#pragma unroll
            for (int i = 0; i < N; ++i) u[i] |= ((x >> i) & 1u) << k;
        }
    }
    int32_t q[N];
    if constexpr (N == 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = from_negabinary(u[i]);
        inv_lift(q[0], q[1], q[2], q[3]);
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) q[perm2(i)] = from_negabinary(u[i]);
#pragma unroll
        for (int x = 0; x < 4; ++x) inv_lift(q[x], q[x + 4], q[x + 8], q[x + 12]);
#pragma unroll
        for (int y = 0; y < 4; ++y) inv_lift(q[4 * y], q[4 * y + 1], q[4 * y + 2], q[4 * y + 3]);
    }
    const float s = ldexpf(1.0f, emax - 30);
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = (float)q[i] * s;
}

template <int NW>
__device__ __forceinline__ void store_words(uint32_t *dst, const uint32_t *w)
{
    if constexpr (NW == 1) dst[0] = w[0];
    else if constexpr (NW == 2) *reinterpret_cast<uint2 *>(dst) = make_uint2(w[0], w[1]);
    else {
#pragma unroll
        for (int i = 0; i < NW / 4; ++i)
            reinterpret_cast<uint4 *>(dst)[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    }
}

template <int NW>
__device__ __forceinline__ void load_words(const uint32_t *src, uint32_t *w)
{
    if constexpr (NW == 1) w[0] = src[0];
    else if constexpr (NW == 2) { const uint2 v = *reinterpret_cast<const uint2 *>(src); w[0] = v.x; w[1] = v.y; }
    else {
#pragma unroll
        for (int i = 0; i < NW / 4; ++i) {
            const uint4 v = reinterpret_cast<const uint4 *>(src)[i];
            w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
        }
    }
}

} // namespace pm
