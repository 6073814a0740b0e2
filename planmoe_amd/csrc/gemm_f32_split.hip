// Batched fp32 GEMM of the expert FFN (experts/ffn.py:63-82 and its backward pass) on gfx950's bf16 matrix cores.
//
// An fp32 value is the sum of three bf16 values: h = bf16(x), m = bf16(x - h), l = x - h - m, each difference exact.  A product of
// two such sums is nine products of bf16 values, each exact in fp32; six of them (hh, hm, mh, hl, mm, lh) hold everything down
// to 2^-26 of the product, less than the rounding of an fp32 product, and are summed in fp32, at 16 times the rate of v_mfma_f32_32x32x2_f32.
// hh has a sum of its own and the five small products another, 2^-8 of it: a matrix core rounds a sum at every instruction, and downwards. All six
// on one sum are six such roundings for 16 k: 0.85 of the fp32 matrix cores' error for N(0, 1) operands, but 1.15 behind a relu, whose zeros
// those add without a rounding, and 1.7 in the column sums of a result, where what is rounded downwards adds up (1 - 3 % of the time for two).
// Against 64 bits, relative 2-norm, fp32 matrix cores and here, k = 512, 1024, 4096: N(0, 1) 4.1e-7, 5.7e-7, 1.15e-6 and 1.3e-7, 1.9e-7, 4.0e-7;
// one operand behind a relu 2.9e-7, 4.1e-7, 8.1e-7 and 1.0e-7, 1.4e-7, 3.2e-7; both positive 3.5e-7, 4.9e-7, 9.9e-7 and 1.3e-7, 1.8e-7, 3.5e-7;
// column sums of 512 rows at k = 1024 5.8e-7 and 2.0e-7.
//
// Eight waves (four in the small tile).  Values come from memory into registers a k-tile of 32 ahead, are split there and go into
// LDS as three planes, either operand with k running fastest whichever way it is stored; two stages, one barrier a k-tile.
// A k-tile is two steps of 16 k: beside the products of the first a wave reads the fragments of the second and splits its share of the next
// k-tile (13 vector instructions a pair of values, 24 values a lane at 256 x 128: 1250 of 3070 clocks of matrix core), beside
// those of the second it reads the first fragments of the next k-tile.
//
// What bounds it: the clock under the matrix cores at 256 x 128 (2 x 4096 x 4096 x 4096: 1317 us = 209 TFLOP/s, 1252 of bf16 products,
// near what gemm_bf16_kernel reaches; 2000 us on the fp32 matrix cores, 137), issuing the splits at 64 x 64.  The two sums fill the registers there
// (251 - 256 of 256, nothing spilt).
#include "gemm_f32_core.hpp"
#include "sp_split.hpp"

namespace pm {

typedef __bf16 sp_bf16x8 __attribute__((ext_vector_type(8)));
typedef uint8_t __attribute__((address_space(3))) *sp_lds;

// WM x WN waves of FM x FN fragments of 32 x 32
template <int WM, int WN, int FM, int FN>
struct SplitShape {
    static constexpr int BM = 32 * FM * WM, BN = 32 * FN * WN, NT = 64 * WM * WN, BK = 32;
    static constexpr int PLANE_A = BM * BK * 2, PLANE_B = BN * BK * 2, STAGE = 3 * (PLANE_A + PLANE_B), LDS = 2 * STAGE;
};

template <int WM, int WN, int FM, int FN, bool TA, bool TB>
__global__ __launch_bounds__((SplitShape<WM, WN, FM, FN>::NT), 2) void gemm_f32_split_kernel(const Gemm32Args p)
{
    using S = SplitShape<WM, WN, FM, FN>;
    constexpr int BM = S::BM, BN = S::BN, NT = S::NT, BK = S::BK, PLANE_A = S::PLANE_A, PLANE_B = S::PLANE_B, STAGE = S::STAGE;
    constexpr int UNITS_A = BM * BK / (8 * NT), UNITS_B = BN * BK / (8 * NT);        // pieces of 8 values of a k-tile that a lane splits
    constexpr int WHOLE = 6 * FM * FN, READS = 3 * (FM + FN);                       // products of a step of 16 k
    extern __shared__ __align__(16) uint8_t lds_bytes[];
    const sp_lds lds = (sp_lds)lds_bytes;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;

    // XCD j (work-groups j, j + 8, ...) takes the j-th eighth of the tiles: batch, panel of 8 columns, row, column
    const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
    const int total = tiles_m * tiles_n * p.batches, per_xcd = (total + 7) / 8;
    const int tile = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per_xcd || tile >= total) return;
    const int e = tile / (tiles_m * tiles_n);
    int in = tile - e * tiles_m * tiles_n;
    const int panel = in / (tiles_m * 8);
    in -= panel * tiles_m * 8;
    const int width = min(8, tiles_n - panel * 8);
    const int m0 = in / width * BM, n0 = (panel * 8 + in % width) * BN;
    int M = p.M, K = p.K;
    if (p.live) {
        int n = 0;
        for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + e];
        n = (n + p.live_round - 1) / p.live_round * p.live_round;
        if (TA) K = min(K, n); else M = min(M, n);
    }
    if (m0 >= M) return;

    const int lda = TA ? p.M : p.K, ldb = TB ? p.N : p.K;
    const uint8_t *A = reinterpret_cast<const uint8_t *>(p.A + (int64_t)e * p.M * p.K + (TA ? (int64_t)m0 : (int64_t)m0 * lda));
    const uint8_t *B = reinterpret_cast<const uint8_t *>(p.B + (int64_t)e * p.N * p.K + (TB ? (int64_t)n0 : (int64_t)n0 * ldb));
    const int64_t ra = TA ? ((int64_t)(K - 1) * lda + (p.M - m0)) * 4 : ((int64_t)(M - m0 - 1) * lda + p.K) * 4;
    const int64_t rb = TB ? ((int64_t)(K - 1) * ldb + (p.N - n0)) * 4 : ((int64_t)(p.N - n0 - 1) * ldb + p.K) * 4;
    const int64_t step_a = TA ? (int64_t)BK * lda * 4 : BK * 4, step_b = TB ? (int64_t)BK * ldb * 4 : BK * 4;
    const int KT = (K + BK - 1) / BK, k_tail = K % BK ? K % BK : BK;
    constexpr uint32_t NOWHERE = 0x80000000u;

    auto desc = [](const uint8_t *base, int64_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, bytes <= 0 ? 0 : bytes > 0x7fffffff ? 0x7fffffff : (int)bytes, 0x00020000);
    };
    // ---- from memory.  k fast: 8 lanes to a row's 128 bytes, quad i of a lane is row tid / 8 + NT / 8 i, k = 4 (tid % 8) ..
    // k slow: lane = column tid % side, eight k each, unit u of a lane is k = 8 (tid / side + NT / side u) ..
    auto fetch = [&](bool T, int side, int ld) -> uint32_t {
        if (T) return ((uint32_t)(8 * (tid / side)) * (uint32_t)ld + (uint32_t)(tid % side)) * 4u;
        return (uint32_t)(tid >> 3) * (uint32_t)ld * 4u + (uint32_t)(tid & 7) * 16u;
    };
    const uint32_t va = fetch(TA, BM, lda), vb = fetch(TB, BN, ldb), past = (tid & 7) * 4 >= k_tail ? NOWHERE : 0u;
    float ga[8 * UNITS_A], gb[8 * UNITS_B];
    auto load_unit = [&](bool T, int side, __amdgpu_buffer_rsrc_t d, uint32_t v, int ld, bool last, int u, float *g) {
        if (T) {
#pragma unroll
            for (int q = 0; q < 8; ++q) g[8 * u + q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(d, v, (uint32_t)(8 * (NT / side) * u + q) * (uint32_t)ld * 4u, 0));
        } else {
            const uint32_t at = v | (last ? past : 0u);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(d, at, (uint32_t)((2 * u + i) * (NT / 8)) * (uint32_t)ld * 4u, 0));
#pragma unroll
                for (int q = 0; q < 4; ++q) g[8 * u + 4 * i + q] = x[q];
            }
        }
    };
    // ---- into LDS: three planes of rows of 64 bytes, the 16 bytes of k = 8 c .. + 7 of row r at unit c ^ (r >> 2) & 3, so that
    // the 16 rows that one pass of a fragment read touches lie at 16 different units of the LDS's 256 bytes
    auto lay_at = [&](bool T, int side, int u) -> uint32_t {
        if (T) { const int r = tid % side, c = tid / side + NT / side * u; return r * 64 + ((c ^ (r >> 2)) & 3) * 16; }
        const int r = (tid >> 3) + 2 * u * (NT / 8), c = (tid & 7) >> 1;
        return r * 64 + ((c ^ (r >> 2)) & 3) * 16 + (tid & 1) * 8;
    };
    const uint32_t la[2] = {lay_at(TA, BM, 0), lay_at(TA, BM, 1)}, lb[2] = {lay_at(TB, BN, 0), lay_at(TB, BN, 1)};
    uint32_t part[3][4];
    // pair x of unit u: split, and stored with the values beside it
    auto split_pair = [&](bool T, int plane, sp_lds to, const uint32_t (&l)[2], int u, int x, const float *g) {
        sp_split(g[8 * u + 2 * x], g[8 * u + 2 * x + 1], part[0][x], part[1][x], part[2][x]);
        if (T) {
            if (x == 3) {
#pragma unroll
                for (int s = 0; s < 3; ++s) *(pm_u32x4 __attribute__((address_space(3))) *)(to + l[u] + s * plane) = pm_u32x4{part[s][0], part[s][1], part[s][2], part[s][3]};
            }
        } else if (x & 1) {
#pragma unroll
            for (int s = 0; s < 3; ++s) *(pm_u32x2 __attribute__((address_space(3))) *)(to + l[u] + (x >> 1) * (NT / 8 * 64) + s * plane) = pm_u32x2{part[s][x - 1], part[s][x]};
        }
    };

    f32x16 acc[FM][FN], low[FM][FN];             // the sums of hh, and of all the others
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = low[i][j][q] = 0.f;
    // ---- fragments: lane = row l % 32, k-chunk l / 32 of the step's 16
    const int fr = lane & 31, fc = lane >> 5;
    uint32_t ro[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) ro[s] = fr * 64 + (((2 * s + fc) ^ (fr >> 2)) & 3) * 16;
    sp_bf16x8 fa[2][3][FM], fb[2][3][FN];                     // [step][part][fragment]
    auto read = [&](sp_lds stage, int s, int x) {
        const int part_ = x / (FM + FN), i = x % (FM + FN);
        if (i < FM) fa[s][part_][i] = *(const sp_bf16x8 __attribute__((address_space(3))) *)(stage + ro[s] + part_ * PLANE_A + 32 * (wm * FM + i) * 64);
        else fb[s][part_][i - FM] = *(const sp_bf16x8 __attribute__((address_space(3))) *)(stage + ro[s] + 3 * PLANE_A + part_ * PLANE_B + 32 * (wn * FN + i - FM) * 64);
    };
    // the small products first (the second operand first: a lane then holds four consecutive columns of one row)
    auto multiply = [&](int s, int x) {
        constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
        const int t = x / (FM * FN), i = x / FN % FM, j = x % FN;
        f32x16 &to = t == 5 ? acc[i][j] : low[i][j];
        to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[s][PB[t]][j], fa[s][PA[t]][i], to, 0, 0, 0);
    };

    constexpr int PAIRS = 4 * (UNITS_A + UNITS_B);
    auto load_tile = [&](int kt) {
        if (kt >= KT) return;
        const auto da = desc(A + kt * step_a, ra - kt * step_a), db = desc(B + kt * step_b, rb - kt * step_b);
        const bool last = kt == KT - 1;
#pragma unroll
        for (int u = 0; u < UNITS_A; ++u) load_unit(TA, BM, da, va, lda, last, u, ga);
#pragma unroll
        for (int u = 0; u < UNITS_B; ++u) load_unit(TB, BN, db, vb, ldb, last, u, gb);
    };
    auto pair = [&](sp_lds to, int n) {
        if (n < 4 * UNITS_A) split_pair(TA, PLANE_A, to, la, n / 4, n % 4, ga);
        else split_pair(TB, PLANE_B, to + 3 * PLANE_A, lb, n / 4 - UNITS_A, n % 4, gb);
    };
    if (KT > 0) {
        load_tile(0);
#pragma unroll
        for (int n = 0; n < PAIRS; ++n) pair(lds, n);
        load_tile(1);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int x = 0; x < READS; ++x) read(lds, 0, x);
    }
    for (int kt = 0; kt < KT; ++kt) {
        const sp_lds here = lds + (kt & 1) * STAGE, next = lds + (~kt & 1) * STAGE;
        // the first 16 k: beside the products, the fragments of the other 16, and the next k-tile's parts into the other stage
        // (behind the last k-tile: what is there once more, not read)
#pragma unroll
        for (int x = 0; x < WHOLE; ++x) {
            multiply(0, x);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = x * 2 * READS / WHOLE; n < (x + 1) * 2 * READS / WHOLE; ++n)
                if (n < READS) read(here, 1, n);
#pragma unroll
            for (int n = x * PAIRS / WHOLE; n < (x + 1) * PAIRS / WHOLE; ++n) pair(next, n);
            __builtin_amdgcn_sched_barrier(0);
        }
        // everybody has read this k-tile to its end and written the next one
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        load_tile(kt + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < WHOLE; ++x) {
            multiply(1, x);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = x * 2 * READS / WHOLE; n < (x + 1) * 2 * READS / WHOLE; ++n)
                if (n < READS) read(next, 0, n);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // An infinity has no parts, nor has what rounds to one: an operand that is not finite, and a sum that overflows, show as a result
    // that is not finite.  Such a wave computes its results again from the values themselves, on the fp32 matrix cores and without LDS (us, all results finite, one
    // column with a NaN, every wave again: 16 x 512, 1024 -> 1024 92, 240, 262; 2 x 4096, 4096 -> 4096 1335, 2805, 3786; 8 x 300, 2048 -> 2048 150, 195, 442).
    float odd = 0.f;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                acc[i][j][q] += low[i][j][q];
                odd = __builtin_fmaf(acc[i][j][q], 0.f, odd);
                acc[i][j][q] *= SP_UNSCALE;
            }
    if (__ballot(odd != odd)) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;
        for (int kt = 0; kt < KT; ++kt) {
            const auto da = desc(A + kt * step_a, ra - kt * step_a), db = desc(B + kt * step_b, rb - kt * step_b);
#pragma unroll 1
            for (int t = 0; t < 4; ++t) {
                const int k = 8 * t + 4 * fc;
                const uint32_t tail = kt * BK + k < K ? 0u : NOWHERE;
                auto quad = [&](bool T, __amdgpu_buffer_rsrc_t d, int row, int ld) {
                    f32x4 v;
                    if (T) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) v[q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(d, ((uint32_t)(k + q) * (uint32_t)ld + (uint32_t)row) * 4u, 0, 0));
                    } else {
                        v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(d, (((uint32_t)row * (uint32_t)ld + (uint32_t)k) * 4u) | tail, 0, 0));
                    }
                    return v;
                };
                f32x4 a[FM], b[FN];
#pragma unroll
                for (int i = 0; i < FM; ++i) a[i] = quad(TA, da, 32 * (wm * FM + i) + fr, lda);
#pragma unroll
                for (int j = 0; j < FN; ++j) b[j] = quad(TB, db, 32 * (wn * FN + j) + fr, ldb);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j][q], a[i][q], acc[i][j], 0, 0, 0);
            }
        }
    }
    g32_store<FM, FN>(p, acc, e, m0, n0, M, wm, wn, m0 / (32 * FM) + wm, (p.M + 64 * FM - 1) / (64 * FM) * 2);
}

template <int WM, int WN, int FM, int FN, bool TA, bool TB>
static int split_launch(const Gemm32Args &p, hipStream_t stream, const char *who)
{
    using S = SplitShape<WM, WN, FM, FN>;
    const auto kernel = gemm_f32_split_kernel<WM, WN, FM, FN, TA, TB>;
    static bool ready[64];                       // (per device; setting the attribute twice does no harm)
    int dev = 0;
    PM_REQUIRE(hipGetDevice(&dev) == hipSuccess, "%s: no device", who);
    if (dev >= 64 || !ready[dev]) {
        PM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS) == hipSuccess,
                   "%s: the kernel needs %d bytes of LDS", who, S::LDS);
        if (dev < 64) ready[dev] = true;
    }
    const int64_t tiles = ((int64_t)p.M + S::BM - 1) / S::BM * (((int64_t)p.N + S::BN - 1) / S::BN) * p.batches;
    PM_REQUIRE(tiles < ((int64_t)1 << 30), "%s: too many tiles", who);
    kernel<<<dim3((unsigned)((tiles + 7) / 8 * 8)), S::NT, S::LDS, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

template <int WM, int WN, int FM, int FN>
static int split_form(int form, const Gemm32Args &p, hipStream_t stream, const char *who)
{
    if (form == 0) return split_launch<WM, WN, FM, FN, false, true>(p, stream, who);
    if (form == 1) return split_launch<WM, WN, FM, FN, false, false>(p, stream, who);
    return split_launch<WM, WN, FM, FN, true, true>(p, stream, who);
}

int gemm_f32_split_run(int form, const Gemm32Args &p, Gemm32Kernel kernel, hipStream_t stream, const char *who)
{
    if (kernel == G32_SPLIT_256) return split_form<4, 2, 2, 2>(form, p, stream, who);
    if (kernel == G32_SPLIT_128) return split_form<2, 4, 2, 1>(form, p, stream, who);
    return split_form<2, 2, 1, 1>(form, p, stream, who);
}

} // namespace pm
