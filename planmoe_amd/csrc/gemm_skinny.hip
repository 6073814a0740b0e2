// The experts' product for few rows: up to 64 rows of an expert against its whole weight, bf16.
//
//   C[e][r][n] = act( bf16( bf16( sum_k A[e][r][k] * B ) + bias[e][n] ) ),  B = B[e][k][n] (nn) or B[e][n][k] (nt)
//
// For experts that have only few rows (decode, small batches).  Bound by reading the weight once, so nothing
// goes through LDS on the way in: a wave loads 16 bytes per lane straight into registers and a work-group's waves (16, or 8 above 32 rows) split the reduction between them, so that a
// compute unit has 128 KB in flight; their sums meet in LDS at the end.  128 columns per work-group.
//   nn: lane = (16 chunks of 8 columns, 4 groups of 8 k): eight loads give an 8 x 8 patch whose columns are
//       put together by byte permutes, each a matrix-core operand of its own (column 8 chunk + c).
//   nt: lane = (16 columns, 4 groups of 16 k): two loads of 8 k, operands as they are; the four groups of a
//       row make 128 consecutive bytes.
// 8 experts x 4 rows, 1024 -> 4096 -> 1024 (67 MB of weights each way): 24 us per product in 128 x 128 tiles.
#include "gemm_skinny.hpp"

namespace pm {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 sk_bf16x8 __attribute__((ext_vector_type(8)));

constexpr int SK_COLS = 128;
constexpr int SK_PITCH = SK_COLS + 4;                       // floats between rows of a wave's 16 x 128 sums in LDS

template <bool NT, int MF, int WAVES, bool GRAD>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_kernel(const SkinnyArgs p)
{
    extern __shared__ __align__(16) float part[];           // [WAVES][16][SK_PITCH]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int e = blockIdx.y, n0 = blockIdx.x * SK_COLS;
    int rows = p.M;
    if (p.live) {
        int n = 0;
        for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + e];
        rows = min(p.M, (n + p.live_round - 1) / p.live_round * p.live_round);
    }
    if (rows == 0 && !(GRAD && p.colsum)) return;

    const uint16_t *A = p.A + (int64_t)e * p.M * p.K;
    const uint16_t *B = p.B + (int64_t)e * p.N * p.K;
    const __amdgpu_buffer_rsrc_t da = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(A), 0, rows > 0 ? rows * p.K * 2 : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(B), 0, (int)((int64_t)p.N * p.K * 2), 0x00020000);
    constexpr uint32_t NOWHERE = 0x80000000u;
    const int l16 = lane & 15, g = lane >> 4;

    f32x4 acc[MF][8];
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[m][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    constexpr int KS = NT ? 64 : 32;                        // k of a step
    const int steps = (p.K + KS - 1) / KS;
    for (int s = wave; s < steps; s += WAVES) {
        if constexpr (!NT) {
            const int k = s * KS + 8 * g;                   // this lane's eight k
            const int col = n0 + 8 * l16;
            pm_u32x4 b[8], a[MF];
            const bool in_n = col < p.N;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                b[q] = __builtin_amdgcn_raw_buffer_load_b128(db, in_n && k + q < p.K ? ((uint32_t)(k + q) * (uint32_t)p.N + (uint32_t)col) * 2u : NOWHERE, 0, 0);
#pragma unroll
            for (int m = 0; m < MF; ++m)
                a[m] = __builtin_amdgcn_raw_buffer_load_b128(da, k < p.K && 16 * m + l16 < rows ? ((uint32_t)(16 * m + l16) * (uint32_t)p.K + (uint32_t)k) * 2u : NOWHERE, 0, 0);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                pm_u32x4 f;
#pragma unroll
                for (int q = 0; q < 4; ++q)                 // column c of rows 2 q and 2 q + 1
                    f[q] = __builtin_amdgcn_perm(b[2 * q + 1][c >> 1], b[2 * q][c >> 1], (c & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
                for (int m = 0; m < MF; ++m)
                    acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sk_bf16x8, a[m]), __builtin_bit_cast(sk_bf16x8, f), acc[m][c], 0, 0, 0);
            }
        } else {
            const int k = s * KS + 16 * g;
            pm_u32x4 b[8][2], a[MF][2];
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int row = n0 + 16 * c + l16;
                    b[c][j] = __builtin_amdgcn_raw_buffer_load_b128(db, row < p.N && k + 8 * j < p.K ? ((uint32_t)row * (uint32_t)p.K + (uint32_t)(k + 8 * j)) * 2u : NOWHERE, 0, 0);
                }
#pragma unroll
            for (int m = 0; m < MF; ++m)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    a[m][j] = __builtin_amdgcn_raw_buffer_load_b128(da, k + 8 * j < p.K && 16 * m + l16 < rows ? ((uint32_t)(16 * m + l16) * (uint32_t)p.K + (uint32_t)(k + 8 * j)) * 2u : NOWHERE, 0, 0);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int c = 0; c < 8; ++c)
#pragma unroll
                    for (int m = 0; m < MF; ++m)
                        acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sk_bf16x8, a[m][j]), __builtin_bit_cast(sk_bf16x8, b[c][j]), acc[m][c], 0, 0, 0);
        }
    }

    // the waves' sums meet in LDS, 16 rows at a time; a lane has rows 4 g .. + 3 of column 8 l16 + c (nn) or 16 c + l16 (nt)
    constexpr int PER = 16 * SK_COLS / (WAVES * 64);        // outputs of a thread: 2 or 4 columns of a row
    const int row_t = tid * PER / SK_COLS, col_t = tid * PER % SK_COLS;
    float *mine = part + wave * 16 * SK_PITCH;
    uint16_t *C = p.C + (int64_t)e * p.M * p.N;
    float colsum = 0.f;                                     // GRAD: of column n0 + tid (tid < 128)
#pragma unroll
    for (int m = 0; m < MF; ++m) {
        if (m > 0) __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float *to = mine + (4 * g + q) * SK_PITCH;
            if constexpr (!NT) {
                *reinterpret_cast<float4 *>(to + 8 * l16) = make_float4(acc[m][0][q], acc[m][1][q], acc[m][2][q], acc[m][3][q]);
                *reinterpret_cast<float4 *>(to + 8 * l16 + 4) = make_float4(acc[m][4][q], acc[m][5][q], acc[m][6][q], acc[m][7][q]);
            } else {
#pragma unroll
                for (int c = 0; c < 8; ++c) to[16 * c + l16] = acc[m][c][q];
            }
        }
        __syncthreads();
        float v[PER];
#pragma unroll
        for (int x = 0; x < PER; ++x) v[x] = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w)
#pragma unroll
            for (int x = 0; x < PER; ++x) v[x] += part[(w * 16 + row_t) * SK_PITCH + col_t + x];
        const int row = 16 * m + row_t, col = n0 + col_t;
        const bool inside = row < rows && col < p.N;        // (N is a multiple of 8: a thread's columns are in or out together)
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            v[x] = bf16_to_f32(f32_to_bf16(v[x]));
            if (!GRAD && p.bias && inside) v[x] = bf16_to_f32(f32_to_bf16(v[x] + bf16_to_f32(p.bias[(int64_t)e * p.N + col + x])));
            if (!GRAD && p.relu) v[x] = v[x] < 0.f ? 0.f : v[x];
            if (GRAD && !(inside && bf16_to_f32(p.mask[((int64_t)e * p.M + row) * p.N + col + x]) > 0.f)) v[x] = 0.f;
        }
        if (inside) {
            uint32_t w[PER / 2];
#pragma unroll
            for (int x = 0; x < PER / 2; ++x) w[x] = f32x2_to_bf16x2(v[2 * x], v[2 * x + 1]);
            uint16_t *to = C + (int64_t)row * p.N + col;
            if constexpr (PER == 4) *reinterpret_cast<uint2 *>(to) = make_uint2(w[0], w[1]);
            else *reinterpret_cast<uint32_t *>(to) = w[0];
        }
        if (GRAD && p.colsum) {
            __syncthreads();
#pragma unroll
            for (int x = 0; x < PER; ++x) part[row_t * SK_PITCH + col_t + x] = v[x];
            __syncthreads();
            if (tid < SK_COLS)
#pragma unroll
                for (int r = 0; r < 16; ++r) colsum += part[r * SK_PITCH + tid];
        }
    }
    if (GRAD && p.colsum && tid < SK_COLS && n0 + tid < p.N) p.colsum[(int64_t)e * p.N + n0 + tid] = colsum;
}

template <bool NT, int MF, int WAVES, bool GRAD>
static int skinny_launch(const SkinnyArgs &p, hipStream_t stream, const char *who)
{
    constexpr int LDS = WAVES * 16 * SK_PITCH * 4;
    const auto kernel = gemm_skinny_kernel<NT, MF, WAVES, GRAD>;
    static bool ready[64];                       // (per device; setting the attribute twice does no harm)
    int dev = 0;
    PM_REQUIRE(hipGetDevice(&dev) == hipSuccess, "%s: no device", who);
    if (dev >= 64 || !ready[dev]) {
        PM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess,
                   "%s: the kernel needs %d bytes of LDS", who, LDS);
        if (dev < 64) ready[dev] = true;
    }
    kernel<<<dim3((unsigned)((p.N + SK_COLS - 1) / SK_COLS), (unsigned)p.batches), WAVES * 64, LDS, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

int gemm_skinny_run(bool nt, SkinnyArgs p, hipStream_t stream, const char *who)
{
    const bool grad = p.mask != nullptr;
#define PM_SK(MF, WAVES_NN, WAVES_NT)                                        \
    (!nt ? skinny_launch<false, MF, WAVES_NN, false>(p, stream, who)         \
     : grad ? skinny_launch<true, MF, WAVES_NT, true>(p, stream, who)        \
            : skinny_launch<true, MF, WAVES_NT, false>(p, stream, who))
    if (p.M <= 16) return PM_SK(1, 16, 16);
    if (p.M <= 32) return PM_SK(2, 16, 8);        // (nt holds 16 KB of weight per step: 8 waves' registers)
    return PM_SK(4, 8, 8);
#undef PM_SK
}

} // namespace pm
