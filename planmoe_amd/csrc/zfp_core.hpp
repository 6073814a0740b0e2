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

// The decoder of 1-D blocks looks at the stream by bit position: the block's words sit in LDS (NW words per
// thread and three zero words behind them: an odd stride) and a look is neighbouring words
// funnel-shifted, so there is no refill state to carry and no branch in the reader.
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

// (zfp's y += w; w = 2 w - y; and the like are a sum and a difference)
__device__ __forceinline__ void inv_lift(int32_t &x, int32_t &y, int32_t &z, int32_t &w)
{
    y += w >> 1; w -= y >> 1;
    auto turn = [](int32_t &a, int32_t &b) { const int32_t t = a; a += b; b -= t; };
    turn(y, w);
    turn(z, x);
    turn(y, z);
    turn(w, x);
}

__device__ __forceinline__ uint32_t to_negabinary(int32_t v) { return ((uint32_t)v + 0xaaaaaaaau) ^ 0xaaaaaaaau; }
__device__ __forceinline__ int32_t from_negabinary(uint32_t v) { return (int32_t)((v ^ 0xaaaaaaaau) - 0xaaaaaaaau); }
// the largest of three, NaN if one of them is (one instruction, v_maximum3_f32)
__device__ __forceinline__ float max3_nan(float a, float b, float c) { return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c); }

// 16 x 16 bit matrix transpose of 16-bit rows, two rows to a word: word j has rows j and j + 8, and afterwards
// columns j and j + 8.  Four exchanges of blocks; the one of 8 x 8 blocks stays inside a word and is a byte permute, done
// where the words are put together (planes_of16) or taken apart (values_of16).  The others are a shift and a bit select a word.
__device__ __forceinline__ uint32_t bit_select(uint32_t m, uint32_t a, uint32_t b) { return (m & a) | (~m & b); }
__device__ __forceinline__ void transpose16_rest(uint32_t (&w)[8])
{
    auto swap_blocks = [](uint32_t &a, uint32_t &b, int s, uint32_t m) {
        const uint32_t t = a >> s;
        a = bit_select(m, a, b << s);
        b = bit_select(m, t, b);
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) swap_blocks(w[j], w[j + 4], 4, 0x0f0f0f0fu);
#pragma unroll
    for (int j = 0; j < 8; ++j) if (!(j & 2)) swap_blocks(w[j], w[j + 2], 2, 0x33333333u);
#pragma unroll
    for (int j = 0; j < 8; j += 2) swap_blocks(w[j], w[j + 1], 1, 0x55555555u);
}
// The bit planes of 16 negabinary values v + 0xaa.. ^ 0xaa.. (u holds v + 0xaa..): their upper 16 or their lower 16 bits, plane k
// (of 16) in half k / 8 of word k % 8; bit i of a plane is value i's.
template <bool HIGH>
__device__ __forceinline__ void planes_of16(const uint32_t (&u)[16], uint32_t (&w)[8])
{
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = __builtin_amdgcn_perm(u[j + 8], u[j], HIGH ? 0x07030602u : 0x05010400u) ^ 0xaaaaaaaau;
    transpose16_rest(w);
}
// and back: upper 16 bits of the values, zeros below
__device__ __forceinline__ void values_of16(uint32_t (&w)[8], uint32_t (&u)[16])
{
    transpose16_rest(w);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        u[j] = __builtin_amdgcn_perm(0u, w[j], 0x02000c0cu);
        u[j + 8] = __builtin_amdgcn_perm(0u, w[j], 0x03010c0cu);
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
// The table holds that expansion for 8 bits of r at a time: entry prev | byte << 1, up to 16 bits, of length
// 8 + prev + ones among the low 7 bits.  What follows the highest
// one (a single '0' test bit, or nothing at the block end) and the implicit last one are a
// matter of the total length, see code16.
__host__ __device__ constexpr uint16_t group_code_entry(int prev, int byte)
{
    uint32_t code = 0; int len = 0;
    for (int p = 0; p < 8; ++p) {
        const int bit = (byte >> p) & 1;
        if (prev) { code |= 1u << len; ++len; }
        code |= (uint32_t)bit << len; ++len;
        prev = bit;
    }
    return (uint16_t)code;
}
struct GroupCodeTable {
    uint16_t entry[512];
    constexpr GroupCodeTable() : entry()
    {
        for (int i = 0; i < 512; ++i) entry[i] = group_code_entry(i & 1, i >> 1);
    }
};
__constant__ const GroupCodeTable group_codes = GroupCodeTable();
// all 256 threads of the work-group; tab has 512 entries
__device__ __forceinline__ void group_code_table(uint16_t *tab)
{
    reinterpret_cast<uint32_t *>(tab)[threadIdx.x] = reinterpret_cast<const uint32_t *>(group_codes.entry)[threadIdx.x];
    __syncthreads();
}

// A block of 4 values; the block's maxbits = 32*NW bits land in bw.
template <int NW>
__device__ __forceinline__ void encode_block4(const float (&f)[4], BitWriter<NW> &bw, uint32_t *lds, const uint16_t *tab)
{
    bw.init(lds);
    const float m = fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fmaxf(fabsf(f[2]), fabsf(f[3])));
    if (!(m > 0.f)) return;                       // all-zero block: '0' flag and zero padding
    // frexp exponent clamped at 1 - 127, i.e. exponent field - 126 (a denormal maximum reads 0)
    const int emax = (int)((__float_as_uint(m) >> 23) & 0xffu) - 126;
    bw.put(2u * (uint32_t)(emax + 127) + 1u, 9);

    // block-floating-point cast: q = (int32)(f * 2^(30 - emax)), x86 conversion on overflow
    const int se = 30 - emax;
    const float s = se > 127 ? INFINITY : __uint_as_float((uint32_t)(se + 127) << 23);
    int32_t q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float v = f[i] * s;
        // -2^31 itself converts to INT_MIN either way
        q[i] = fabsf(v) < 2147483648.0f ? (int32_t)v : (int32_t)0x80000000;
    }
    fwd_lift(q[0], q[1], q[2], q[3]);
    uint32_t u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = to_negabinary(q[i]);

    // embedded coding: bit planes from the top, group-tested, until the budget is spent
    int bits = 32 * NW - 9;
    int nsig = 0;
    for (int k = 31; k >= 0 && bits > 0; --k) {
        uint32_t x = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) x |= ((u[i] >> k) & 1u) << i;
        const int mm = min(nsig, bits);
        bits -= mm;
        bw.put(x & ((1u << mm) - 1u), mm);
        if (nsig < 4 && bits > 0) {
            const uint32_t r = x >> mm;                   // mm == nsig here
            // r == 0 runs through the same formulas: top = -1, no code bits, length 1 (the '0')
            const int top = 31 - __clz((int)r), ones = __builtin_popcount(r);
            // cut after the highest one bit (not emitted when it is the block's last value),
            // then one more '0' test bit unless the block ends there
            const int lt = top + 1 + ones - (nsig + top == 3);
            const int emit = min(lt + (nsig + top < 3 ? 1 : 0), bits);
            bw.put(tab[r * 2u + 1u] & ((1u << min(lt, emit)) - 1u), emit);
            bits -= emit;
            nsig += top + 1;
        }
    }
    bw.finish();
}

// A block of 4 x 4 values, in registers throughout.
//   PACK  s: its maxbits = 32 * NW bits.  They come in from above: what a plane adds (31 bits at most: the verbatim bits of nsig
//         values, then at most two for each of the others less one) shifts the whole down by its length, a funnel shift a
//         word, and what the budget cuts off never comes in.  (Bits gathered in a register pair and stored to LDS word by word took two
//         such appends a plane and a dozen instructions each.)
//   TRIP  f: what the decoder makes of those bits, where the block's largest value is finite (else f is as it was; see zfp_trip16).
//         It has the planes that fit whole, and the cut one as far as its bits are there.
// Returns the exponent field of the largest magnitude.
template <int NW, bool PACK, bool TRIP>
__device__ __forceinline__ int code16(float (&f)[16], uint32_t *s, const uint16_t *tab)
{
    if constexpr (PACK) {
#pragma unroll
        for (int i = 0; i < NW; ++i) s[i] = 0u;
    }
    // the largest magnitude, NaN if there is one
    float m = fabsf(f[0]);
#pragma unroll
    for (int i = 1; i < 15; i += 2) m = max3_nan(m, fabsf(f[i]), fabsf(f[i + 1]));
    m = max3_nan(m, fabsf(f[15]), fabsf(f[15]));
    int field = (int)(__float_as_uint(m) >> 23);
    int32_t q[16];
    // block-floating-point cast: q = (int32)(f * 2^(30 - emax)), x86 conversion on overflow: only where the factor itself is
    // none (next to the denormals) or a value is not finite is there any
    if (__builtin_amdgcn_ballot_w64((uint32_t)(field - 29) > 225u && m != 0.f) != 0) {
        m = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) m = fmaxf(m, fabsf(f[i]));
        field = (int)(__float_as_uint(m) >> 23);
        const int se = 156 - field;
        const float scale = se > 127 ? INFINITY : __uint_as_float((uint32_t)(se + 127) << 23);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float v = f[i] * scale;
            // -2^31 itself converts to INT_MIN either way
            q[i] = !(m > 0.f) ? 0 : fabsf(v) < 2147483648.0f ? (int32_t)v : (int32_t)0x80000000;
        }
    } else {
        const float scale = __uint_as_float((uint32_t)(283 - max(field, 29)) << 23);
#pragma unroll
        for (int i = 0; i < 16; ++i) q[i] = (int32_t)(f[i] * scale);
    }
    // all zero: a '0' and zeros behind it
    const bool live = m > 0.f;
    int bits = live ? 32 * NW - 9 : 0, nsig = 0;
    // the flag and the exponent, frexp's clamped at 1 - 127, i.e. the field - 126 (a denormal maximum reads 0) and biased by 127.  That of an
    // infinity has a bit too many, which gets into the first plane's.
    const uint32_t head = live ? 2u * (uint32_t)(field + 1) + 1u : 0u;
    if constexpr (PACK) s[NW - 1] = head << 23;

#pragma unroll
    for (int y = 0; y < 4; ++y) fwd_lift(q[4 * y], q[4 * y + 1], q[4 * y + 2], q[4 * y + 3]);
#pragma unroll
    for (int x = 0; x < 4; ++x) fwd_lift(q[x], q[x + 4], q[x + 8], q[x + 12]);
    uint32_t u[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) u[i] = (uint32_t)q[perm2(i)] + 0xaaaaaaaau;

    // Embedded coding: bit planes from the top, group-tested, until the budget is spent.  A plane is nsig bits as they are; then the
    // group tests: a bit for every value up to the highest one, a test bit in front of the first and behind every one, where the last
    // of them ends the plane (the block's last value: its one is implied, no test behind it).
    bool whole = live;                            // (TRIP) every plane so far fits
    int cut = -1;                                 // the plane that does not, from which on bits and nsig stay
    uint32_t cut_plane = 0u;
    auto plane = [&](uint32_t x, int k) __attribute__((always_inline)) {
        const uint32_t r = x >> nsig, r1 = 2u * r + 1u;       // (a one in front: the table's index, and never zero)
        const int top = 31 - __builtin_clz(r1), next = nsig + top, ones = __builtin_popcount(r);
        const int coded = top + ones, need = max(coded + (next < 16 ? 1 : -1), 0);
        const int total = nsig + need;
        if constexpr (PACK) {
            const uint32_t lo = tab[r1 & 0x1ffu], hi = tab[r1 >> 8];
            const uint32_t code = lo | (hi << (9 + __builtin_popcount(r & 0x7fu)));
            uint32_t v = __builtin_amdgcn_ubfe(x, 0u, nsig) | (__builtin_amdgcn_ubfe(code, 0u, min(coded, need)) << nsig);
            if (k == 31) v |= head >> 9;
            const int emit = TRIP && !whole ? 0 : min(total, bits);
#pragma unroll
            for (int i = 0; i < NW - 1; ++i) s[i] = __builtin_amdgcn_alignbit(s[i + 1], s[i], emit);
            s[NW - 1] = __builtin_amdgcn_alignbit(v, s[NW - 1], emit);
            if constexpr (!TRIP) { bits -= emit; nsig = next; }
        }
        if constexpr (TRIP) {
            cut_plane = whole ? x : cut_plane;
            cut = whole ? k : cut;
            whole = whole && total <= bits;
            bits = whole ? bits - total : bits;
            nsig = whole ? next : nsig;
        }
    };
    auto more = [&]() { return __builtin_amdgcn_ballot_w64(TRIP ? whole : bits > 0) != 0; };        // (a branch of the whole wave)
    uint32_t w[8];
    planes_of16<true>(u, w);
#pragma unroll
    for (int k = 15; k >= 0; --k) if (more()) plane(k < 8 ? w[k] & 0xffffu : w[k - 8] >> 16, k + 16);
    if (more()) {
        planes_of16<false>(u, w);
#pragma unroll
        for (int k = 15; k >= 0; --k) if (more()) plane(k < 8 ? w[k] & 0xffffu : w[k - 8] >> 16, k);
    }
    if constexpr (PACK) {
        // (32 planes and bits to spare)
        for (int left = TRIP && !whole ? 0 : bits; left > 0; left -= 31) {
            const int n = min(left, 31);
#pragma unroll
            for (int i = 0; i < NW - 1; ++i) s[i] = __builtin_amdgcn_alignbit(s[i + 1], s[i], n);
            s[NW - 1] >>= n;
        }
    }
    if constexpr (TRIP) {
        if (field == 255) return field;
#pragma unroll
        for (int i = 0; i < 16; ++i) u[i] ^= 0xaaaaaaaau;
        if (live && !whole) {
            // what the decoder makes of the bits that are there: a run of zeros that the budget cuts short ends in a one
            int n = nsig, b = bits;
            const int mm = min(n, b);
            uint32_t x = cut_plane & ((1u << mm) - 1u);
            b -= mm;
            while (n < 16 && b > 0) {
                --b;
                const uint32_t r = cut_plane >> n;
                if (r == 0u) break;
                const int z = __builtin_ctz(r), lim = min(15 - n, b);
                b -= z < lim ? z + 1 : lim;
                n += min(z, lim);
                x |= 1u << n;
                ++n;
            }
            const uint32_t above = ~((2u << cut) - 1u);
#pragma unroll
            for (int i = 0; i < 16; ++i) u[i] = (u[i] & above) | (((x >> i) & 1u) << cut);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) q[perm2(i)] = from_negabinary(u[i]);
#pragma unroll
        for (int x = 0; x < 4; ++x) inv_lift(q[x], q[x + 4], q[x + 8], q[x + 12]);
#pragma unroll
        for (int y = 0; y < 4; ++y) inv_lift(q[4 * y], q[4 * y + 1], q[4 * y + 2], q[4 * y + 3]);
        const float back = ldexpf(1.0f, field - 156);
#pragma unroll
        for (int i = 0; i < 16; ++i) f[i] = (float)q[i] * back;
    }
    return field;
}

// ---- group tests of a 2-D block's bit plane, eleven stream bits at a time
// The group-test bits of a plane are a walk with two states: a test bit is due (T), or the zeros of
// a run up to the next one bit are being read (R).  walk16_step is what eleven stream bits do to it from state T on, as if there were values
// without end: in bits 0..9 the one bits found (relative to the first value that was not significant), in 10..13 the values passed, one
// more in state R (the value being read), in 14 whether it ends in R, in 15 whether it goes on.  A walk that goes on in state R goes on in T
// with a test bit in front.  Where the block's last value is reached its one is implied and the plane ends, and how many bits
// a plane took follows from its values: its own for each, and a test bit for each one and the end.
__host__ __device__ constexpr uint16_t walk16_step(uint32_t bits)
{
    int n = 0, used = 0;
    uint32_t ones = 0;
    while (used < 11) {
        if (!((bits >> used++) & 1u)) return (uint16_t)(ones | ((uint32_t)n << 10));
        while (true) {
            if (used == 11) return (uint16_t)(ones | ((uint32_t)(n + 1) << 10) | 0xc000u);
            if ((bits >> used++) & 1u) break;
            ++n;
        }
        ones |= 1u << n++;
    }
    return (uint16_t)(ones | ((uint32_t)n << 10) | 0x8000u);
}
constexpr int WALK16_ENTRIES = 2048;
struct Walk16Table {
    uint16_t step[WALK16_ENTRIES];
    constexpr Walk16Table() : step()
    {
        for (int i = 0; i < WALK16_ENTRIES; ++i) step[i] = walk16_step((uint32_t)i);
    }
};
__constant__ const Walk16Table walk16_table __attribute__((aligned(16))) = Walk16Table();

// all 256 threads of the work-group copy the table into LDS (4 KB); a barrier follows
__device__ __forceinline__ void walk16_load(uint16_t *tab)
{
    reinterpret_cast<uint4 *>(tab)[threadIdx.x] = reinterpret_cast<const uint4 *>(walk16_table.step)[threadIdx.x];
    __syncthreads();
}

// One bit plane of a 2-D block, bit by bit as zfp walks it: look = the next 32 stream bits (a plane
// never uses more than 31), bits = what is left of the block's budget, nsig = values significant so
// far.  nsig verbatim bits, then segment by segment the test bit and the zeros up to the next one
// bit (cut short by the budget or by the block's last value, whose one is implied).
__device__ __forceinline__ uint32_t slow_plane16(uint32_t look, int &bits, int &nsig)
{
    constexpr int N = 16;
    const int mm = min(nsig, bits);
    bits -= mm;
    uint32_t x = look & ((1u << mm) - 1u);
    look >>= mm;
    while (nsig < N && bits > 0) {
        if (!(look & 1u)) { --bits; break; }
        const int lim = min(N - 1 - nsig, bits - 1);
        const uint32_t win = (look >> 1) & ((1u << lim) - 1u);
        const int z = win != 0u ? __builtin_ctz(win) : lim;       // zeros read
        const int used = 1 + (win != 0u ? z + 1 : lim);
        look >>= used; bits -= used; nsig += z;
        x |= 1u << nsig;
        ++nsig;
    }
    return x;
}

// A block of 4 values
template <int NW>
__device__ __forceinline__ void decode_block4(BitReader<NW> &br, float (&f)[4])
{
    if (!br.get(1)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = 0.f;
        return;
    }
    const int emax = (int)br.get(8) - 127;
    uint32_t u[4] = {0u, 0u, 0u, 0u};
    int bits = 32 * NW - 9;
    int nsig = 0;
    for (int k = 31; k >= 0 && bits > 0; --k) {
        const int mm = min(nsig, bits);
        bits -= mm;
        uint32_t x = br.get(mm);
        while (nsig < 4 && bits > 0) {
            // tiny blocks: test bit and run are read separately (measured faster here)
            --bits;
            if (!br.get(1)) break;
            const int lim = min(3 - nsig, bits);
            const uint32_t win = br.peek() & ((1u << lim) - 1u);
            const int z = win != 0u ? __builtin_ctz(win) : lim;
            const int used = win != 0u ? z + 1 : lim;
            br.skip(used); bits -= used; nsig += z;
            x |= 1u << nsig;
            ++nsig;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] |= ((x >> i) & 1u) << k;
    }
    int32_t q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = from_negabinary(u[i]);
    inv_lift(q[0], q[1], q[2], q[3]);
    const float s = ldexpf(1.0f, emax - 30);
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = (float)q[i] * s;
}

// A block of 4 x 4 values from its NW words s, which are shifted down as planes are read; tab: the table above.
template <int NW>
__device__ __forceinline__ void decode16(uint32_t (&s)[NW], float (&f)[16], const uint16_t *tab)
{
    auto skip = [&](int n) __attribute__((always_inline)) {          // n <= 31
#pragma unroll
        for (int i = 0; i < NW - 1; ++i) s[i] = __builtin_amdgcn_alignbit(s[i + 1], s[i], n);
        s[NW - 1] >>= n;
    };
    const uint32_t head = s[0];
    skip(9);
    int bits = 32 * NW - 9, nsig = 0, cut = -1;
    // A lane reads planes by table up to the one that the budget ends in (there is one in nearly every block): bits, nsig and the
    // stream stay as they are there, and it is walked bit by bit afterwards, by all lanes at once.
    bool whole = (head & 1u) != 0u;
    // planes 31..16 are collected as rows and transposed into the coefficients' upper halves
    uint32_t w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = 0u;
#pragma unroll
    for (int k = 15; k >= 0; --k) {
        if (whole) {
            uint32_t x = __builtin_amdgcn_ubfe(s[0], 0u, nsig), look = s[0] >> nsig;
            int at = nsig, next;
            while (true) {
                const uint32_t e = tab[look & (WALK16_ENTRIES - 1)];
                x |= (e & 0x3ffu) << at;
                next = at + (int)__builtin_amdgcn_ubfe(e, 10u, 4u);
                if (e < 0x8000u || next > 15) break;
                const int reading = (int)__builtin_amdgcn_ubfe(e, 14u, 1u);
                look = (look >> (11 - reading)) | (uint32_t)reading;
                at = next - reading;
            }
            next = min(next, 16);
            const int total = next + __builtin_popcount((x & 0x7fffu) >> nsig) + (next < 16);
            x = (x & 0xffffu) | (next == 16 && nsig < 16 ? 0x8000u : 0u);
            whole = total <= bits;
            if (whole) {
                w[k & 7] |= x << (16 * (k >> 3));
                bits -= total;
                nsig = next;
                skip(total);
            } else {
                cut = k;
            }
        }
    }
    int cut_bits = bits, cut_nsig = nsig;
    if (cut >= 0) {
        const uint32_t x = slow_plane16(s[0], cut_bits, cut_nsig) << (16 * (cut >> 3));
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] |= (cut & 7) == j ? x : 0u;
    }
    uint32_t u[16];
    values_of16(w, u);
    if (whole)
        for (int k = 15; k >= 0 && bits > 0; --k) {
            const int before = bits;
            const uint32_t x = slow_plane16(s[0], bits, nsig);
            skip(before - bits);
#pragma unroll
            for (int i = 0; i < 16; ++i) u[i] |= ((x >> i) & 1u) << k;
        }
    int32_t q[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) q[perm2(i)] = from_negabinary(u[i]);
#pragma unroll
    for (int x = 0; x < 4; ++x) inv_lift(q[x], q[x + 4], q[x + 8], q[x + 12]);
#pragma unroll
    for (int y = 0; y < 4; ++y) inv_lift(q[4 * y], q[4 * y + 1], q[4 * y + 2], q[4 * y + 3]);
    // (a block without a stream has values of zero: zeros whatever the factor, which is finite)
    const float scale = ldexpf(1.0f, (int)((head >> 1) & 0xffu) - 157);
#pragma unroll
    for (int i = 0; i < 16; ++i) f[i] = (float)q[i] * scale;
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
