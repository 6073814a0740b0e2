// The experts' weight gradients where an expert has few rows: C[e][m][n] = sum_k A[e][k][m] * B[e][k][n], bf16 or fp32, k the rows in use.
//
// Bound by writing C.  A wave takes 32 rows by 64 columns (bf16: 128, or 256) on its own, operands from memory straight into registers, no LDS and no
// barrier: it has nothing to wait for but its few loads, and what it stores is 256 bytes of a row at a time (a lane's columns are next to each
// other: fragment j of the second operand is every J-th column from the j-th on).  The tiles of the other kernels load a whole k-tile of 32
// or 64, pass it through LDS and, in fp32, store 32 bytes of a row at a time, two or three of them on a compute unit.
// fp32 as in gemm_f32_split.hip, in three bf16 parts, the sums in the same order: the same bits where operands and sums are finite.  A wave with one that is not
// sums its 32 x 64 again in another order, the tiles theirs, so that what is finite beside it may differ in its last bits.
//
// us, the tiles and this:
//   fp32  16 x 1 row, 3328 x 3072 204, 98    8 x 8, 2600 x 3440 94, 56    16 x 2, 1896 x 688 31, 18    8 x 2, 4096 x 4096 162, 81    8 x 64, 2048 x 2048 59, 45
//   bf16  16 x 1 row, 3328 x 3072  85, 53    8 x 8, 2600 x 3440 54, 31    8 x 29, 1888 x 1256 17, 12   8 x 2, 4096 x 4096  67, 42    8 x 64, 2048 x 2048 22, 18
//
// Stored past the caches: an optimizer reads a weight gradient once and late.  Rows that are not whole lines share a line with the next row's wave, which
// the caches put together: such rows are stored plainly, in bf16 256 columns a wave so that there are fewer of those lines, in fp32 only where the last
// cache (256 MB) does not hold the result.  In bf16 the waves that share lines are brought together as well (8 experts x 8 rows, 2600 x 3440, 37 and 31 us; in fp32 16 x 1,
// 3328 x 3072 103 and 117).  Neither a step of k asked for ahead of the products nor 128 rows of 64 columns a work-group gained anything in the others.  What that choice
// is from, us, before the waves were brought together: 32 x 128 (bf16 256) plain and past the caches, 32 x 64 (bf16 128) plain and past them; of these fp32 has the last two, bf16 the
// first and the last, the others were not kept
//   fp32  16 x 1, 3328 x 3072  119, 116, 134, 112     8 x 8, 2600 x 3440    56, 58, 56, 63     16 x 2, 1896 x 688   23, 22, 20, 19
//         8 x 2, 4096 x 4096   94, 84, 108, 89        8 x 64, 2048 x 2048   52, 50, 50, 50     8 x 128, 2048 x 2048 81, 80, 85, 83
//         4 x 128, 512 x 1024  14.8, 13.5, 10.9, 10.3
//   bf16  16 x 1, 3328 x 3072  63, 65, 61, 59         8 x 8, 2600 x 3440    38, 41, 42, 48     16 x 2, 1896 x 688   12, 12, 16, 16
//         8 x 2, 4096 x 4096   57, 55, 45, 43         8 x 64, 2048 x 2048   27, 25, 22, 18     8 x 80, 2048 x 2048  29, 27, 24, 22
//         8 x 64, 1896 x 1032  17, 17, 17, 16         8 x 100, 2048 x 2048  32, 31, 29, 27
#include "gemm_outer.hpp"
#include "sp_split.hpp"

namespace pm {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 op_bf16x8 __attribute__((ext_vector_type(8)));

template <bool F32, int J, bool NT>
__global__ __launch_bounds__(256, !F32 && J == 8 ? 2 : 4) void gemm_outer_kernel(const OuterArgs p)
{
    constexpr int COLS = 32 * J, SIZE = F32 ? 4 : 2, W = J * SIZE / 4;        // W: words of a lane's columns
    typedef uint32_t words __attribute__((ext_vector_type(W)));
    constexpr uint32_t NOWHERE = 0x80000000u;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 31, fc = lane >> 5;
    // The waves of a work-group lie next to each other; DOWN: one below the other, and XCD j (work-groups j, j + 8, ...) takes the j-th eighth, so that what shares a
    // line of C shares an L2
    constexpr bool DOWN = !F32 && J == 8;
    constexpr int BELOW = DOWN ? 4 : 1, BESIDE = 4 / BELOW;
    const int groups_n = (p.N + BESIDE * COLS - 1) / (BESIDE * COLS), groups_m = (p.M + 32 * BELOW - 1) / (32 * BELOW), total = groups_n * groups_m * p.batches;
    const int number = DOWN ? blockIdx.x % 8 * ((total + 7) / 8) + blockIdx.x / 8 : blockIdx.x;
    if (number >= total || (DOWN && (int)blockIdx.x / 8 >= (total + 7) / 8)) return;
    const int e = number / (groups_n * groups_m), in = number - e * groups_n * groups_m;
    const int m0 = (in / groups_n * BELOW + (DOWN ? wave : 0)) * 32, n0 = (in % groups_n * BESIDE + (DOWN ? 0 : wave)) * COLS;
    if (n0 >= p.N || m0 >= p.M) return;
    int K = p.K;
    if (p.live) {
        int n = 0;
        for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + e];
        K = min(K, (n + p.live_round - 1) / p.live_round * p.live_round);
    }
    const char *A = (const char *)p.A + (int64_t)e * p.K * p.M * SIZE, *B = (const char *)p.B + (int64_t)e * p.K * p.N * SIZE;
    const __amdgpu_buffer_rsrc_t da = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(A), 0, p.K * p.M * SIZE, 0x00020000);
    const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(B), 0, p.K * p.N * SIZE, 0x00020000);
    // a lane's row of C, and its J columns in a row (N is a multiple of J: in or out together)
    const int row = m0 + c, col = n0 + J * c;
    auto at_a = [&](int k) { return k < K && row < p.M ? ((uint32_t)k * (uint32_t)p.M + (uint32_t)row) * SIZE : NOWHERE; };
    auto at_b = [&](int k) { return k < K && col < p.N ? ((uint32_t)k * (uint32_t)p.N + (uint32_t)col) * SIZE : NOWHERE; };

    f32x16 acc[J], low[F32 ? J : 1];             // fp32: the sums of the upper parts' products, and of all the others
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int q = 0; q < 16; ++q) { acc[j][q] = 0.f; if (F32) low[F32 ? j : 0][q] = 0.f; }
    // a step of 16 k: lane = row (columns) c, k = 8 fc .. + 7
    words b[8];
    uint32_t a[8];
    auto load_b = [&](int k) {
        if constexpr (W == 4) return __builtin_bit_cast(words, __builtin_amdgcn_raw_buffer_load_b128(db, at_b(k), 0, 0));
        else return __builtin_bit_cast(words, __builtin_amdgcn_raw_buffer_load_b64(db, at_b(k), 0, 0));
    };
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (F32) a[i] = __builtin_amdgcn_raw_buffer_load_b32(da, at_a(k0 + 8 * fc + i), 0, 0);
            else a[i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(da, at_a(k0 + 8 * fc + i), 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) b[i] = load_b(k0 + 8 * fc + i);
    };
    for (int k0 = 0; k0 < K; k0 += 16) {
        load(k0);
        if constexpr (F32) {
            constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};        // the small products first
            pm_u32x4 fa[3];
            auto split = [&](float x0, float x1, pm_u32x4 (&f)[3], int x) {
                uint32_t h, m, l;
                sp_split(x0, x1, h, m, l);
                f[0][x] = h; f[1][x] = m; f[2][x] = l;
            };
#pragma unroll
            for (int x = 0; x < 4; ++x) split(__uint_as_float(a[2 * x]), __uint_as_float(a[2 * x + 1]), fa, x);
#pragma unroll
            for (int j = 0; j < J; ++j) {
                pm_u32x4 fb[3];
#pragma unroll
                for (int x = 0; x < 4; ++x) split(__uint_as_float(b[2 * x][j % W]), __uint_as_float(b[2 * x + 1][j % W]), fb, x);
#pragma unroll
                for (int t = 0; t < 6; ++t) {
                    f32x16 &to = t == 5 ? acc[j] : low[F32 ? j : 0];
                    to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(op_bf16x8, fa[PA[t]]), __builtin_bit_cast(op_bf16x8, fb[PB[t]]), to, 0, 0, 0);
                }
            }
        } else {
            pm_u32x4 fa, fb[J];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                fa[x] = a[2 * x] | a[2 * x + 1] << 16;
#pragma unroll
                for (int j = 0; j < J; ++j) fb[j][x] = __builtin_amdgcn_perm(b[2 * x + 1][j / 2 % W], b[2 * x][j / 2 % W], j & 1 ? 0x07060302u : 0x05040100u);
            }
#pragma unroll
            for (int j = 0; j < J; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(op_bf16x8, fa), __builtin_bit_cast(op_bf16x8, fb[j]), acc[j], 0, 0, 0);
        }
    }
    if constexpr (F32) {
        // (an operand that is not finite, or a sum that overflows, has no parts: from the values themselves, see gemm_f32_split.hip)
        float odd = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                acc[j][q] += low[F32 ? j : 0][q];
                odd = __builtin_fmaf(acc[j][q], 0.f, odd);
                acc[j][q] *= SP_UNSCALE;
            }
        if (__ballot(odd != odd)) {
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[j][q] = 0.f;
#pragma unroll 1
            for (int k0 = 0; k0 < K; k0 += 8)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float x = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(da, at_a(k0 + 4 * fc + q), 0, 0));
                    const words y = load_b(k0 + 4 * fc + q);
#pragma unroll
                    for (int j = 0; j < J; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, __uint_as_float(y[j % W]), acc[j], 0, 0, 0);
                }
        }
    }
    // a lane has rows 8 q + 4 fc .. + 3 of its columns in acc[.][4 q ..]
    char *to = (char *)p.C + ((int64_t)e * p.M * p.N + (int64_t)m0 * p.N + n0) * SIZE;
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(to, 0, (int)min((int64_t)0x7fffffff, ((int64_t)(p.M - m0 - 1) * p.N + (p.N - n0)) * SIZE), 0x00020000);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int r = (q >> 2) * 8 + 4 * fc + (q & 3);
        words v;
#pragma unroll
        for (int x = 0; x < W; ++x) v[x] = F32 ? __float_as_uint(acc[x][q]) : f32x2_to_bf16x2(acc[2 * x % J][q], acc[(2 * x + 1) % J][q]);
        const uint32_t at = col < p.N && m0 + r < p.M ? ((uint32_t)r * (uint32_t)p.N + (uint32_t)(J * c)) * SIZE : NOWHERE;
        if constexpr (W == 4) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(pm_u32x4, v), out, at, 0, NT ? 2 : 0);
        else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(pm_u32x2, v), out, at, 0, NT ? 2 : 0);
    }
}

template <bool F32, int J, bool NT>
static int outer_launch(const OuterArgs &p, hipStream_t stream, const char *who)
{
    const int64_t down = !F32 && J == 8 ? 128 : 32, across = !F32 && J == 8 ? 32 * J : 128 * J;          // a work-group's
    const int64_t blocks = ((int64_t)p.M + down - 1) / down * (((int64_t)p.N + across - 1) / across) * p.batches;
    gemm_outer_kernel<F32, J, NT><<<dim3((unsigned)((blocks + 7) / 8 * 8)), 256, 0, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

// Up to 100 rows in fp32 and 64 in bf16, whose tiles take less for a row; an expert may have half as many again.  Fewer where the result has few waves, whose steps of 16
// rows are a trip to memory each, and in bf16 where rows are not whole lines.  us, the tiles and this
//   bf16  5 x 264 x 520, 33 rows 4.4, 5.0;  4 x 256 x 256, 24 rows 4.4, 3.8;  4, 40 and 64 rows
//         8 x 512 x 512 5.9, 3.8   5.9, 5.3   6.1, 6.8   8 x 1024 x 1024 10.0, 6.0   10.1, 6.8   10.1, 8.0   16 x 1024 x 1032 16.7, 10.5   17.0, 14.8   17.5, 18.8
//   fp32  4, 40 and 100 rows  8 x 264 x 520 5.5, 5.1   6.6, 6.9   8.6, 10.8  8 x 512 x 512     6.1, 5.0    7.3, 6.7    9.4, 10.7  8 x 1024 x 1024  15.1, 8.9    18.1, 12.7   22.3, 20.4
bool gemm_outer_serves(int dtype, int m, int n, int64_t k, int batches, int64_t rows)
{
    const int64_t size = dtype == PLANMOE_F32 ? 4 : 2, values = (int64_t)m * n * batches;
    const bool large = values > (int64_t)4 << 20;
    const int64_t most = dtype == PLANMOE_F32 ? large ? 100 : values > (int64_t)3 << 19 ? 48 : 8
                                                        : large && (int64_t)n * size % 128 == 0 ? 64 : values > (int64_t)3 << 19 ? 40 : 24;
    return rows <= most && 2 * k <= 3 * most && k * m * size < ((int64_t)1 << 31) && k * n * size < ((int64_t)1 << 31) &&
           ((int64_t)m + 31) / 32 * (((int64_t)n + 255) / 256) * batches < ((int64_t)1 << 30);
}

int gemm_outer_run(int dtype, const OuterArgs &p, hipStream_t stream, const char *who)
{
    const int64_t row = (int64_t)p.N * (dtype == PLANMOE_F32 ? 4 : 2);
    const bool lines = row % 128 == 0;
    if (dtype == PLANMOE_F32)
        return lines || row * p.M * p.batches <= (int64_t)256 << 20 ? outer_launch<true, 2, true>(p, stream, who) : outer_launch<true, 2, false>(p, stream, who);
    return lines ? outer_launch<false, 4, true>(p, stream, who) : outer_launch<false, 8, false>(p, stream, who);
}

} // namespace pm
