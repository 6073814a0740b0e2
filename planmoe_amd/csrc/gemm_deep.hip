// The experts' product where there are few tiles: 128 x 128 with four k-tiles of 64 in LDS, or 128 x 64 with five, bf16.
//
//   C[e][m][n] = act( bf16( bf16( sum_k A[e][m][k] * B[e][n][k] ) + bias[e][n] ) ), either operand stored k fast or k slow
//
// A wave of gemm_bf16_kernel's 128 x 128 tile reads for one phase of four products while it works on the phase before, so each phase ends in
// waiting for LDS: 0.5 us a k-tile on a compute unit of its own, 0.21 of it matrix core.  Here a wave's fragments are read three steps of 16 k
// ahead, with one barrier a k-tile; a load or a read goes between every two products, places in LDS are constants (the loop is as many k-tiles long as LDS holds), and
// one descriptor serves an operand.  Four waves, two by two, each 64 x 64 (64 x 32); one work-group per compute unit and tile.
#include "gemm_deep.hpp"

namespace pm {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 dp_bf16x8 __attribute__((ext_vector_type(8)));
typedef short dp_s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t dp_u32x4 __attribute__((ext_vector_type(4)));
typedef const uint8_t __attribute__((address_space(3))) *dp_lds;

constexpr int DP_BK = DEEP_BK, DP_SIDE = 128, DP_OPERAND = DP_SIDE * DP_BK * 2;        // (A's k-tile in LDS)

// k-tiles in LDS: 128 KB, or 120 with 64 columns
constexpr int dp_stages(int J) { return J == 2 ? 4 : 5; }

// (ds_read_b64_tr_b16 hands a lane four consecutive k of its column, see gemm.hip)
__device__ __forceinline__ dp_bf16x8 dp_read_tr(dp_lds lo, dp_lds hi)
{
    typedef dp_s16x4 __attribute__((address_space(3))) *tr;
    const dp_s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr)lo), y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr)hi);
    return __builtin_bit_cast(dp_bf16x8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
}

// SHARES: of the work-groups of a tile each takes a share of the k-tiles and leaves its sums, in fp32, in a plane of its own
// J: 32-column fragments of a wave; the tile is 128 x 64 J
template <int J, bool TA, bool TB, bool GRAD, bool SHARES = false>
__global__ __launch_bounds__(256, 1) void gemm_deep_kernel(const SkinnyArgs p)
{
    constexpr int DP_STAGES = dp_stages(J), DP_COLS = 64 * J, OPERAND_B = DP_COLS * DP_BK * 2, LOADS = 4 + 2 * J;        // loads: of a wave for a k-tile
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

    // XCD j (work-groups j, j + 8, ...) takes the j-th eighth of the tiles: batch, panel of 8 columns, row, column
    const int tiles_m = (p.M + DP_SIDE - 1) / DP_SIDE, tiles_n = (p.N + DP_COLS - 1) / DP_COLS;
    const int total = tiles_m * tiles_n * p.batches * (SHARES ? p.splits : 1), per_xcd = (total + 7) / 8;
    int tile = blockIdx.x % 8 * per_xcd + blockIdx.x / 8, share = 0;
    if (blockIdx.x / 8 >= per_xcd || tile >= total) return;
    if (SHARES) {                                // (the share before the tile: an XCD's work-groups are at the same k)
        const int tiles = tiles_m * tiles_n * p.batches;
        share = tile / tiles;
        tile -= share * tiles;
    }
    const int e = tile / (tiles_m * tiles_n);
    int in = tile - e * tiles_m * tiles_n;
    const int panel = in / (tiles_m * 8);
    in -= panel * tiles_m * 8;
    const int width = min(8, tiles_n - panel * 8);
    const int m0 = in / width * DP_SIDE, n0 = (panel * 8 + in % width) * DP_COLS;
    int M = p.M, K = p.K;
    if (p.live) {
        int n = 0;
        for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + e];
        n = (n + p.live_round - 1) / p.live_round * p.live_round;
        if (TA) K = min(K, n); else M = min(M, n);
    }
    if (m0 >= M) return;

    const int lda = TA ? p.M : p.K, ldb = TB ? p.N : p.K;
    const uint16_t *A = p.A + (int64_t)e * p.M * p.K + (TA ? (int64_t)m0 : (int64_t)m0 * lda);
    const uint16_t *B = p.B + (int64_t)e * p.N * p.K + (TB ? (int64_t)n0 : (int64_t)n0 * ldb);
    if (SHARES) {
        const int each = ((K + DP_BK - 1) / DP_BK + p.splits - 1) / p.splits * DP_BK, k0 = min(share * each, K);
        A += TA ? (int64_t)k0 * lda : k0;
        B += TB ? (int64_t)k0 * ldb : k0;
        K = min(each, K - k0);
    }
    auto desc = [](const void *base, int64_t bytes) {
        const uint64_t a = (uint64_t)base;
        return dp_u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes <= 0 ? 0u : bytes > 0x7fffffff ? 0x7fffffffu : (uint32_t)bytes, 0x00020000u};
    };
    const dp_u32x4 da = desc(A, TA ? ((int64_t)(K - 1) * lda + (p.M - m0)) * 2 : ((int64_t)(M - m0 - 1) * lda + K) * 2);
    const dp_u32x4 db = desc(B, TB ? ((int64_t)(K - 1) * ldb + (p.N - n0)) * 2 : ((int64_t)(p.N - n0 - 1) * ldb + K) * 2);
    const int KT = __builtin_amdgcn_readfirstlane((K + DP_BK - 1) / DP_BK), last = KT > 0 ? KT - 1 : 0, k_tail = K % DP_BK ? K % DP_BK : DP_BK;
    constexpr uint32_t NOWHERE = 0x80000000u;

    // ---- which 16 bytes a lane fetches.  k fast: 128 rows of 128 bytes, a load fills eight, chunk c of row r at unit c ^ (r >> 1) & 7.
    // k slow: 64 rows of 256 bytes, a load fills four, chunk c of row k at unit c ^ (k & 3) << 2; of 128 bytes, eight, c ^ (k >> 1 & 1) << 2.
    auto fetch = [&](bool T, int X, int i, int ld) -> uint32_t {        // X: 64 X rows (columns)
        if (T && X == 1) return (uint32_t)(16 * wave + (lane >> 3)) * (uint32_t)ld * 2u + (uint32_t)((lane & 7) ^ (((lane >> 4) & 1) << 2)) * 16u;
        if (T) return (uint32_t)(16 * wave + (lane >> 4)) * (uint32_t)ld * 2u + (uint32_t)((lane & 15) ^ (((lane >> 4) & 3) << 2)) * 16u;
        const int row = 16 * X * wave + 8 * i + (lane >> 3);
        return (uint32_t)row * (uint32_t)ld * 2u + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    };
    const uint32_t va[2] = {fetch(TA, 2, 0, lda), fetch(TA, 2, TA ? 0 : 1, lda)}, vb[2] = {fetch(TB, J, 0, ldb), fetch(TB, J, TB ? 0 : 1, ldb)};
    // (chunks of a k-fast row past the end of K are asked for out of range)
    auto past = [&](int i) -> uint32_t { return (int)(((lane & 7) ^ ((4 * i + (lane >> 4)) & 7)) * 8) >= k_tail ? NOWHERE : 0u; };
    const uint32_t past0 = past(0), past1 = past(1);
    // the n-th of a k-tile's.  Past the end the last k-tile is asked for again, so that the count of what is on its way stays the same.
    auto load = [&](int kt, int stage, int n) {
        const bool b = n >= 4, T = b ? TB : TA, end = kt == KT - 1 && k_tail != DP_BK;
        const int i = b ? n - 4 : n, X = b ? J : 2;
        const uint32_t ld = (uint32_t)(b ? ldb : lda), v = (b ? vb[i & 1] : va[i & 1]) | (!T && end ? ((i & 1) ? past1 : past0) : 0u);
        const uint32_t soff = __builtin_amdgcn_readfirstlane(ld * 2u * (uint32_t)(T ? 8 / X * i : 8 * (i & ~1)) + (uint32_t)(kt < KT ? kt : last) * (T ? ld * (DP_BK * 2u) : DP_BK * 2u));
        const uint32_t to = lds0 + (b ? DP_STAGES * DP_OPERAND + stage * OPERAND_B : stage * DP_OPERAND) + wave * (X * 2048) + i * 1024;
        asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(to), "v"(v), "s"(b ? db : da), "s"(soff) : "memory", "m0");
    };

    // ---- fragments: 32 rows (columns) x 16 k; lane = row l % 32, k-chunk l / 32
    const int fr = lane & 31, fc = lane >> 5, tg = lane >> 4, ts = lane & 15;
    auto place = [&](bool T, int X, int n, int w) -> uint32_t {     // k fast: step n; k slow: fragment n
        if (T) {
            const int row = 8 * (tg >> 1) + (ts >> 2), c = 4 * X * w + 4 * n + 2 * (tg & 1) + ((ts & 3) >> 1);
            return row * (128 * X) + (X == 2 ? c ^ ((ts >> 2) << 2) : c ^ ((ts >> 3) << 2)) * 16 + 8 * (ts & 1);
        }
        return (32 * X * w + fr) * 128 + (((2 * n + fc) ^ ((fr >> 1) & 7)) * 16);
    };
    uint32_t ra[4], rb[4];
#pragma unroll
    for (int n = 0; n < (TA ? 2 : 4); ++n) ra[n] = lds0 + place(TA, 2, n, wm);
#pragma unroll
    for (int n = 0; n < (TB ? J : 4); ++n) rb[n] = lds0 + DP_STAGES * DP_OPERAND + place(TB, J, n, wn);
    dp_bf16x8 fa[4][2], fb[4][J];                // [step][fragment]
    auto read = [&](int stage, int s, int x) {   // x: A's fragments 0, 1, B's
        const bool b = x >= 2, T = b ? TB : TA;
        const int i = x & 1, X = b ? J : 2, at = stage * (b ? OPERAND_B : DP_OPERAND);
        dp_bf16x8 f;
        if (T) {
            const dp_lds q = (dp_lds)(uintptr_t)(b ? rb[i] : ra[i]) + at + s * (16 * 128 * X);
            f = dp_read_tr(q, q + 4 * 128 * X);
        } else {
            f = *(const dp_bf16x8 __attribute__((address_space(3))) *)((dp_lds)(uintptr_t)(b ? rb[s] : ra[s]) + at + i * 4096);
        }
        if (b) fb[s][i] = f; else fa[s][i] = f;
    };

    f32x16 acc[2][J];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;

#pragma unroll
    for (int kt = 0; kt < DP_STAGES - 1; ++kt)
#pragma unroll
        for (int n = 0; n < LOADS; ++n) load(kt, kt, n);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((DP_STAGES - 2) * LOADS) : "memory");
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int x = 0; x < 2 + J; ++x) read(0, s, x);
    for (int k0 = 0; k0 < KT; k0 += DP_STAGES) {
#pragma unroll
        for (int stage = 0; stage < DP_STAGES; ++stage) {
            const int kt = k0 + stage;
            if (kt >= KT) break;
            // behind the barrier everybody's share of k-tile kt + 1 is in, and everybody is done with kt - 1
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((DP_STAGES - 3) * LOADS) : "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int x = 0; x < 2 * J; ++x) {
                    const int i = x / J, j = x % J;
                    // (the second operand first: a lane then holds four consecutive columns of one row)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[s][j], fa[s][i], acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    // the step before this one's registers get what comes three steps on: this k-tile's last step, or the next one's first three
                    auto next = [&](int y) { if (s == 0) read(stage, 3, y); else read((stage + 1) % DP_STAGES, s - 1, y); };
                    next(x);
                    if (J == 1 && x == 0) next(2);
                    const int q = 2 * J * s + x;             // (J = 1: six loads under eight products)
                    if (J == 2 ? q & 1 : q & 3) load(kt + DP_STAGES - 1, (stage + DP_STAGES - 1) % DP_STAGES, J == 2 ? q >> 1 : q - 1 - (q >> 2));
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
    }

    // ---- a lane has row fr of fragment i, columns 8 q + 4 fc .. + 3 of fragment j in acc[i][j][4 q ..]
    if constexpr (SHARES) {
        float *plane = p.shares + ((int64_t)(share * p.batches + e) * p.M + m0) * p.N + n0;
        const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(plane, 0, (int)min((int64_t)0x7fffffff, ((int64_t)(M - m0 - 1) * p.N + (p.N - n0)) * 4), 0x00020000);
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int col = 32 * J * wn + 32 * j + 8 * q + 4 * fc;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int row = 64 * wm + 32 * i + fr;
                    const pm_u32x4 v = {__float_as_uint(acc[i][j][4 * q]), __float_as_uint(acc[i][j][4 * q + 1]), __float_as_uint(acc[i][j][4 * q + 2]), __float_as_uint(acc[i][j][4 * q + 3])};
                    __builtin_amdgcn_raw_buffer_store_b128(v, to, n0 + col < p.N ? ((uint32_t)row * (uint32_t)p.N + (uint32_t)col) * 4u : NOWHERE, 0, 0);
                }
            }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }
    const int64_t corner = (int64_t)e * p.M * p.N + (int64_t)m0 * p.N + n0;
    const int bytes = (int)min((int64_t)0x7fffffff, ((int64_t)(M - m0 - 1) * p.N + (p.N - n0)) * 2);
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(p.C + corner, 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t mask = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(GRAD ? p.mask + corner : p.C), 0, GRAD ? bytes : 0, 0x00020000);
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int col = 32 * J * wn + 32 * j + 8 * q + 4 * fc;
            const bool in_n = n0 + col < p.N;    // (N is a multiple of 8: a lane's columns are in or out together)
            float add[4] = {0.f, 0.f, 0.f, 0.f}, sums[4] = {0.f, 0.f, 0.f, 0.f};
            if (!GRAD && p.bias && in_n)
#pragma unroll
                for (int x = 0; x < 4; ++x) add[x] = bf16_to_f32(p.bias[(int64_t)e * p.N + n0 + col + x]);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = 64 * wm + 32 * i + fr;
                const uint32_t at = in_n ? ((uint32_t)row * (uint32_t)p.N + (uint32_t)col) * 2u : NOWHERE;
                uint32_t v[2];
#pragma unroll
                for (int x = 0; x < 2; ++x) v[x] = f32x2_to_bf16x2(acc[i][j][4 * q + 2 * x], acc[i][j][4 * q + 2 * x + 1]);
                if (!GRAD && p.bias) {           // the matmul's rounding is done; torch.add in bf16
#pragma unroll
                    for (int x = 0; x < 2; ++x) v[x] = f32x2_to_bf16x2(__uint_as_float(v[x] << 16) + add[2 * x], __uint_as_float(v[x] & 0xffff0000u) + add[2 * x + 1]);
                }
                if (!GRAD && p.relu) {
#pragma unroll
                    for (int x = 0; x < 2; ++x) v[x] = relu_bf16x2(v[x]);
                }
                if (GRAD) {                      // relu's backward: kept where its output was positive
                    const pm_u32x2 keep = __builtin_bit_cast(pm_u32x2, __builtin_amdgcn_raw_buffer_load_b64(mask, at, 0, 0));
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        v[x] &= ((int)(keep[x] << 16) > 0 ? 0xffffu : 0u) | ((int)keep[x] >= 0x10000 ? 0xffff0000u : 0u);
                        sums[2 * x] += __uint_as_float(v[x] << 16);
                        sums[2 * x + 1] += __uint_as_float(v[x] & 0xffff0000u);
                    }
                }
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(pm_u32x2, make_uint2(v[0], v[1])), out, at, 0, 0);
            }
            if (GRAD && p.colsum) {              // (rows past M: their mask reads as zero)
#pragma unroll
                for (int x = 0; x < 4; ++x)
#pragma unroll
                    for (int d = 1; d < 32; d <<= 1) sums[x] += __shfl_xor(sums[x], d);
                const int slots = tiles_m * 2, slot = m0 / DP_SIDE * 2 + wm;
                if (fr == 0 && in_n) *reinterpret_cast<float4 *>(p.colsum + ((int64_t)e * slots + slot) * p.N + n0 + col) = make_float4(sums[0], sums[1], sums[2], sums[3]);
            }
        }
    // nothing may still be on its way into LDS that another work-group gets
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int J, bool TA, bool TB, bool GRAD, bool SHARES = false>
static int deep_launch(const SkinnyArgs &p, hipStream_t stream, const char *who)
{
    constexpr int DP_LDS = dp_stages(J) * (DP_OPERAND + 64 * J * DP_BK * 2);
    const auto kernel = gemm_deep_kernel<J, TA, TB, GRAD, SHARES>;
    static bool ready[64];                       // (per device; setting the attribute twice does no harm)
    int dev = 0;
    PM_REQUIRE(hipGetDevice(&dev) == hipSuccess, "%s: no device", who);
    if (dev >= 64 || !ready[dev]) {
        PM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, DP_LDS) == hipSuccess,
                   "%s: the kernel needs %d bytes of LDS", who, DP_LDS);
        if (dev < 64) ready[dev] = true;
    }
    const int64_t tiles = ((int64_t)p.M + DP_SIDE - 1) / DP_SIDE * (((int64_t)p.N + 64 * J - 1) / (64 * J)) * p.batches * (SHARES ? p.splits : 1);
    PM_REQUIRE(tiles < ((int64_t)1 << 30), "%s: too many tiles", who);
    kernel<<<dim3((unsigned)((tiles + 7) / 8 * 8)), 256, DP_LDS, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

int gemm_deep_shares_run(const SkinnyArgs &p, hipStream_t stream, const char *who) { return deep_launch<2, false, true, false, true>(p, stream, who); }

bool gemm_deep_reaches(int form, int m, int n, int64_t k)
{
    const int64_t reach = ((int64_t)1 << 31) / 2;
    return (form == 1 || (k + 256) * n < reach) && (form != 2 || (k + 256) * m < reach);
}

template <int J>
static int deep_run(int form, const SkinnyArgs &p, hipStream_t stream, const char *who)
{
    if (form == 0) return deep_launch<J, false, true, false>(p, stream, who);
    if (form == 2) return deep_launch<J, true, true, false>(p, stream, who);
    return p.mask ? deep_launch<J, false, false, true>(p, stream, who) : deep_launch<J, false, false, false>(p, stream, who);
}
int gemm_deep_run(int form, int columns, const SkinnyArgs &p, hipStream_t stream, const char *who)
{
    return columns == 64 ? deep_run<1>(form, p, stream, who) : deep_run<2>(form, p, stream, who);
}

} // namespace pm
