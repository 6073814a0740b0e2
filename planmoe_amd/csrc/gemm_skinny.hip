// The experts' product for few rows: up to 32 rows of an expert against its whole weight, bf16.
//
//   C[e][r][n] = act( bf16( bf16( sum_k A[e][r][k] * B ) + bias[e][n] ) ),  B = B[e][k][n] (nn) or B[e][n][k] (nt)
//
// For experts that have only few rows (decode, small batches).  Bound by reading the weight once, so nothing
// goes through LDS on the way in: a wave loads straight into registers, a work-group's waves (16, or 8 where
// registers ask for it) split the reduction between them, one to eight steps each in flight, so that a compute unit has
// 128 or 256 KB on its way; the waves' sums meet in LDS at the end.
//   nn: lane = (16 chunks of C columns, 4 groups of 8 k): eight loads give an 8 x C patch whose columns are
//       put together by byte permutes, each a matrix-core operand of its own (column C chunk + c).
//   nt: lane = (16 columns, 4 groups of 16 k): two loads of 8 k, operands as they are; the four groups of a
//       row make 128 consecutive bytes.
// 8 experts x 2 rows, 67 MB of weights that no cache holds (a plain read of them takes 11.5 - 14): 1024 -> 4096 14.8 -> 13.5 us with
// nontemporal loads, 4096 -> 1024 22.9 -> 18.5 in 32 columns, b^T 20.3 -> 14.3 (128 x 128 tiles: 41 us).  Loads of the next steps go out
// while a step is worked on: 4 x 20 rows, 4096 -> 4096 b^T 33.6 -> 28.1 (all of a wave's steps at once, then none until they are used).
#include "gemm_skinny_core.hpp"

namespace pm {

// MF: 16-row fragments; C: 16-column fragments of the weight, a work-group's columns / 16; U: steps of the reduction a wave has in flight;
// LARGE: the weight does not stay in the caches anyway (skinny_large): read nontemporally (nt: not, the two loads of 128 bytes meet in the cache; nn in
// 32 columns: not, two work-groups' halves of a line do)
// SHARES: a grid of (column groups, batches that can have rows, shares of the reduction); the y-th batch is the y-th that has rows
template <bool NT, int MF, int C, int U, int WAVES, bool GRAD, bool LARGE, bool SHARES = false>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_kernel(const SkinnyArgs p)
{
    extern __shared__ __align__(16) float part[];           // [WAVES][16][16 C + 4]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int e, n0, rows = p.M;
    if constexpr (SHARES) {
        int n = 0;
        if (lane < p.batches)
            for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + lane];
        n = min(p.M, (n + p.live_round - 1) / p.live_round * p.live_round);
        uint64_t used = __ballot(n > 0);
        if ((int)blockIdx.y >= __popcll(used)) return;
        for (int y = blockIdx.y; y > 0; --y) used &= used - 1;
        e = __builtin_ctzll(used);
        rows = __builtin_amdgcn_readlane(n, e);
        n0 = blockIdx.x * 16 * C;
    } else {
        skinny_tile<16 * C, C == 2 && (LARGE || !NT)>(e, n0);
    }
    if (!SHARES && p.live) {
        int n = 0;
        for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + e];
        rows = min(p.M, (n + p.live_round - 1) / p.live_round * p.live_round);
    }
    if (rows == 0 && !(GRAD && p.colsum)) return;

    const uint16_t *A = p.A + (int64_t)e * p.M * p.K;
    const uint16_t *B = p.B + (int64_t)e * p.N * p.K;
    const __amdgpu_buffer_rsrc_t da = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(A), 0, rows > 0 ? rows * p.K * 2 : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(B), 0, (int)((int64_t)p.N * p.K * 2), 0x00020000);
    constexpr uint32_t NOWHERE = SK_NOWHERE;
    const int l16 = lane & 15, g = lane >> 4;

    f32x4 acc[MF][C];
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int c = 0; c < C; ++c) acc[m][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    constexpr int KS = NT ? 64 : 32;                        // k of a step
    int steps = (p.K + KS - 1) / KS, first = wave;          // of this wave: first, first + WAVES, .. below steps
    if constexpr (SHARES) {
        const int each = (steps + p.splits - 1) / p.splits;
        first += blockIdx.z * each;
        steps = min(steps, (int)(blockIdx.z + 1) * each);
    }
    const uint32_t place = n0 + C * l16 < p.N ? ((uint32_t)(8 * g) * (uint32_t)p.N + (uint32_t)(n0 + C * l16)) * 2u : NOWHERE;    // (nn)
    // U steps of the wave are on their way: a step's loads go out as soon as the registers of the step U before it are free
    auto walk = [&](auto load, auto use) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (first + u * WAVES < steps) load(u, first + u * WAVES);
        for (int s0 = first; s0 < steps; s0 += U * WAVES) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (s0 + u * WAVES < steps) use(u);
                if (s0 + (U + u) * WAVES < steps) load(u, s0 + (U + u) * WAVES);
            }
        }
    };
    if constexpr (!NT) {
        SkinnyWeights<C, LARGE> b[U];
        pm_u32x4 a[U][MF];
        walk([&](int u, int s) {
            const int k = s * KS + 8 * g;                   // this lane's eight k
            b[u].load(db, place, s, p.N);
#pragma unroll
            for (int m = 0; m < MF; ++m)
                a[u][m] = __builtin_amdgcn_raw_buffer_load_b128(da, k < p.K && 16 * m + l16 < rows ? ((uint32_t)(16 * m + l16) * (uint32_t)p.K + (uint32_t)k) * 2u : NOWHERE, 0, 0);
        }, [&](int u) { b[u].multiply(a[u], acc); });
    } else {
        pm_u32x4 b[U][C][2], a[U][MF][2];
        walk([&](int u, int s) {
            const int k = s * KS + 16 * g;
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int row = n0 + 16 * c + l16;
                    b[u][c][j] = __builtin_amdgcn_raw_buffer_load_b128(db, row < p.N && k + 8 * j < p.K ? ((uint32_t)row * (uint32_t)p.K + (uint32_t)(k + 8 * j)) * 2u : NOWHERE, 0, 0);
                }
#pragma unroll
            for (int m = 0; m < MF; ++m)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    a[u][m][j] = __builtin_amdgcn_raw_buffer_load_b128(da, k + 8 * j < p.K && 16 * m + l16 < rows ? ((uint32_t)(16 * m + l16) * (uint32_t)p.K + (uint32_t)(k + 8 * j)) * 2u : NOWHERE, 0, 0);
        }, [&](int u) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int c = 0; c < C; ++c)
#pragma unroll
                    for (int m = 0; m < MF; ++m)
                        acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sk_bf16x8, a[u][m][j]), __builtin_bit_cast(sk_bf16x8, b[u][c][j]), acc[m][c], 0, 0, 0);
        });
    }

    skinny_finish<NT, MF, C, WAVES, GRAD, SHARES>(p, e, n0, rows, acc, part);
}

template <bool NT, int MF, int C, int U, int WAVES, bool GRAD, bool LARGE, bool SHARES = false>
static int skinny_launch(const SkinnyArgs &p, hipStream_t stream, const char *who)
{
    constexpr int COLS = 16 * C, LDS = WAVES * 16 * (COLS + 4) * 4;
    const auto kernel = gemm_skinny_kernel<NT, MF, C, U, WAVES, GRAD, LARGE, SHARES>;
    static bool ready[64];                       // (per device; setting the attribute twice does no harm)
    int dev = 0;
    PM_REQUIRE(hipGetDevice(&dev) == hipSuccess, "%s: no device", who);
    if (dev >= 64 || !ready[dev]) {
        PM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess,
                   "%s: the kernel needs %d bytes of LDS", who, LDS);
        if (dev < 64) ready[dev] = true;
    }
    kernel<<<dim3((unsigned)((p.N + COLS - 1) / COLS), (unsigned)(SHARES ? p.active : p.batches), (unsigned)(SHARES ? p.splits : 1)), WAVES * 64, LDS, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

// From 16 MB on a weight is read past the caches; below, the next call may find it there (us, plain and nontemporal: 8 experts x 2,
// 512 -> 512 4.0, 5.2; 4 x 2, 1024 -> 1024 4.7, 5.6; 8 x 2, 1024 -> 1024 6.8, 6.8; 16 x 2, 1024 -> 1024 8.8, 7.9).  What a model's other layers
// have pushed out of the last cache (256 MB) gains by it; a weight that the same call read before loses: 8 x 8, 2048 -> 2048 in 64
// columns 16.6, 14.6 cold and 11.9, 12.7 in the cache; 16 x 8, 1024 -> 4096 27.8, 25.5 and 21.9, 24.2.
bool skinny_large(int64_t n, int64_t k, int64_t batches) { return n * k * batches * 2 >= (int64_t)16 << 20; }

// Columns of a work-group: 32 or 64 where that leaves a compute unit for each work-group (one compute unit gets at most 28 GB/s
// from memory, however much it has on its way); else the width that takes a compute unit through the fewest columns, 128 where two
// widths do (nn in 96, whose pieces of a row are 12 bytes, is no faster than in 128).
// us with cold weights (every one of 1.6 GB in turn), rows in use of 8 and 24, in 32, 64, 96 and 128 columns:
//   8 experts x 2, 1024 -> 4096         nn 23, 14.5, -, 13.5      nt 15, 14, -, 13.8
//   8 x 2, 4096 -> 1024                 nn 18.5, 20.4, -, 27      nt 14.3, 20, -, 30
//   8 x 2, 3072 -> 1536                 nn 28, 17.1, -, 24        nt 19, 16.5, -, 24          (384, 192, 96 work-groups)
//   4 x 2, 4096 -> 512                  nn 16.4, 18.3, -, 24      nt 11, 19, -, 26
//   8 x 20, 4096 -> 1024                nn 22.4, 25, -, 35        nt 17.4, 24, -, 43
//   8 x 8, 2688 -> 2560                 nn 37, 30, 29, 23         nt 24, 33, 23, 29
// (nn in 32 columns reads 64 bytes of a row, two work-groups a line: it takes the compute units that 64 leave idle, but no more.  Not nontemporally, or
// the second of them finds its half gone.  us in 64 columns, in 32 nontemporal and in 32, weights in the last cache and cold:
//   8 x 8, 4096 -> 1024    13.9, 18.2, 14.5    23.9, 20.0, 20.8      4 x 8, 4096 -> 1024    12.4, 13.5, 10.9    21.1, 18.6, 19.1
//   8 x 24, same           17.6, 22.9, 16.6    27.8, 23.9, 24.2      8 x 8, 3072 -> 768     12.0, 11.6, 9.0     17.4, 13.8, 14.0
//   8 x 8, 8192 -> 512     23.2, 32.8, 21.3    39.4, 35.2, 34.9      16 x 8, 8192 -> 256    22.5, 29.1, 18.8    34.6, 30.8, 31.0)
int gemm_skinny_run(bool nt, SkinnyArgs p, hipStream_t stream, const char *who)
{
    const bool grad = p.mask != nullptr, large = skinny_large(p.N, p.K, p.batches);
#define PM_SK_NN(MF, C, U, WAVES) (large ? skinny_launch<false, MF, C, U, WAVES, false, true>(p, stream, who)                    \
                                         : skinny_launch<false, MF, C, U, WAVES, false, false>(p, stream, who))
#define PM_SK_NT(MF, C, U, WAVES, LARGE) (grad ? skinny_launch<true, MF, C, U, WAVES, true, LARGE>(p, stream, who)               \
                                               : skinny_launch<true, MF, C, U, WAVES, false, LARGE>(p, stream, who))
    const int width = gemm_skinny_width(nt, p.N, p.K, p.batches);
    const bool few = p.M <= 16;
    if (!nt) {
        if (width == 32) return few ? skinny_launch<false, 1, 2, 8, 16, false, false>(p, stream, who) : skinny_launch<false, 2, 2, 8, 8, false, false>(p, stream, who);
        if (width == 64) return few ? PM_SK_NN(1, 4, 2, 16) : PM_SK_NN(2, 4, 2, 16);
        return few ? PM_SK_NN(1, 8, 1, 16) : PM_SK_NN(2, 8, 1, 16);
    }
    // (12 or 16 KB of weight per step: with 17 rows and more 8 waves' registers)
    switch (width) {
    case 32:
        if (large) return few ? PM_SK_NT(1, 2, 2, 16, true) : PM_SK_NT(2, 2, 4, 8, true);
        return few ? PM_SK_NT(1, 2, 2, 16, false) : PM_SK_NT(2, 2, 4, 8, false);
    case 64: return few ? PM_SK_NT(1, 4, 1, 16, false) : PM_SK_NT(2, 4, 1, 16, false);
    case 96: return few ? PM_SK_NT(1, 6, 1, 16, false) : PM_SK_NT(2, 6, 1, 8, false);
    default: return few ? PM_SK_NT(1, 8, 1, 16, false) : PM_SK_NT(2, 8, 1, 8, false);
    }
#undef PM_SK_NN
#undef PM_SK_NT
}

int gemm_skinny_shares_run(const SkinnyArgs &p, hipStream_t stream, const char *who)
{
    const bool large = skinny_large(p.N, p.K, p.active);
    if (p.M <= 16) return large ? skinny_launch<false, 1, 4, 2, 16, false, true, true>(p, stream, who) : skinny_launch<false, 1, 4, 2, 16, false, false, true>(p, stream, who);
    return large ? skinny_launch<false, 2, 4, 2, 16, false, true, true>(p, stream, who) : skinny_launch<false, 2, 4, 2, 16, false, false, true>(p, stream, who);
}

int gemm_skinny_width(bool nt, int n, int64_t k, int batches)
{
    const int64_t cu = compute_units();
    auto groups = [&](int width) { return (int64_t)((n + width - 1) / width) * batches; };
    auto columns = [&](int width) { return (groups(width) + cu - 1) / cu * width; };
    if (groups(32) <= cu && (nt || skinny_large(n, k, batches))) return 32;        // (nn, small: 4.0 us in 64 columns, 5.2 in 32)
    if (groups(64) <= cu) return 64;
    if (!nt) return 128;
    if (columns(128) <= columns(64) && columns(128) <= columns(96)) return 128;
    return columns(96) <= columns(64) ? 96 : 64;
}

} // namespace pm
