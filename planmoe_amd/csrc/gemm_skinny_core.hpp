// What the kernels for few rows are made of: the weight's loads, a step's products, and the end of the sums.
#pragma once
#include "gemm_skinny.hpp"

namespace pm {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 sk_bf16x8 __attribute__((ext_vector_type(8)));

constexpr uint32_t SK_NOWHERE = 0x80000000u;                // an offset that is out of any descriptor's range

// Expert and first column of a work-group of a grid of (column groups, experts).
// PAIRS: neighbours in columns (nn: they share lines of 128 bytes) are, of every 16 work-groups, i and i + 8, which go to one XCD.
template <int COLS, bool PAIRS>
__device__ __forceinline__ void skinny_tile(int &e, int &n0)
{
    int group = blockIdx.x;
    e = blockIdx.y;
    if (PAIRS) {
        const int id = e * gridDim.x + group, in = id % 16, first = id - in;
        const int at = first + 16 <= (int)(gridDim.x * gridDim.y) ? first + 2 * (in % 8) + in / 8 : id;
        e = at / gridDim.x;
        group = at % gridDim.x;
    }
    n0 = group * COLS;
}

// nn: a lane's eight k of C columns.  Its place in a step of 32 k stays, the step and the row are the scalar offset: K is a multiple of 8, so
// a lane's eight k are inside or the descriptor's business together.
// ONCE: nontemporal
template <int C, bool ONCE>
struct SkinnyWeights {
    typedef uint32_t row __attribute__((ext_vector_type(C / 2)));
    row b[8];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t d, uint32_t place, int step, int N)
    {
        const uint32_t at = (uint32_t)step * 64u * (uint32_t)N;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if constexpr (C == 8) b[q] = __builtin_amdgcn_raw_buffer_load_b128(d, place, at + (uint32_t)(q * 2) * (uint32_t)N, ONCE ? 2 : 0);
            else if constexpr (C == 4) b[q] = __builtin_amdgcn_raw_buffer_load_b64(d, place, at + (uint32_t)(q * 2) * (uint32_t)N, ONCE ? 2 : 0);
            else b[q][0] = __builtin_amdgcn_raw_buffer_load_b32(d, place, at + (uint32_t)(q * 2) * (uint32_t)N, ONCE ? 2 : 0);
        }
    }
    template <int MF>
    __device__ __forceinline__ void multiply(const pm_u32x4 (&a)[MF], f32x4 (&acc)[MF][C]) const
    {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            pm_u32x4 f;
#pragma unroll
            for (int q = 0; q < 4; ++q)                     // column c of rows 2 q and 2 q + 1
                f[q] = __builtin_amdgcn_perm(b[2 * q + 1][c >> 1], b[2 * q][c >> 1], (c & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
            for (int m = 0; m < MF; ++m)
                acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sk_bf16x8, a[m]), __builtin_bit_cast(sk_bf16x8, f), acc[m][c], 0, 0, 0);
        }
    }
};

// SHARES: the sums as they are, into this work-group's share
template <bool NT, int MF, int C, int WAVES, bool GRAD, bool SHARES = false>
__device__ __forceinline__ void skinny_finish(const SkinnyArgs &p, int e, int n0, int rows, const f32x4 (&acc)[MF][C], float *part)
{
    constexpr int SK_COLS = 16 * C, SK_PITCH = SK_COLS + 4;             // (floats between rows of a wave's sums in LDS)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    // the waves' sums meet in LDS, 16 rows at a time; a lane has rows 4 g .. + 3 of column C l16 + c (nn) or 16 c + l16 (nt)
    constexpr int EACH = (16 * SK_COLS + WAVES * 64 - 1) / (WAVES * 64), PER = EACH == 3 ? 4 : EACH;        // outputs of a thread: 1, 2 or 4 columns of a row
    const bool writes = tid * PER < 16 * SK_COLS;           // (96 columns: three threads in four)
    const int row_t = writes ? tid * PER / SK_COLS : 0, col_t = tid * PER % SK_COLS;
    float *mine = part + wave * 16 * SK_PITCH;
    uint16_t *out = p.C + (int64_t)e * p.M * p.N;
    float colsum = 0.f;                                     // GRAD: of column n0 + tid
#pragma unroll
    for (int m = 0; m < MF; ++m) {
        if (m > 0) __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float *to = mine + (4 * g + q) * SK_PITCH;
            if constexpr (!NT) {
#pragma unroll
                for (int c = 0; c + 4 <= C; c += 4)
                    *reinterpret_cast<float4 *>(to + C * l16 + c) = make_float4(acc[m][c][q], acc[m][c + 1][q], acc[m][c + 2][q], acc[m][c + 3][q]);
                if constexpr (C == 2) *reinterpret_cast<float2 *>(to + 2 * l16) = make_float2(acc[m][0][q], acc[m][1][q]);
            } else {
#pragma unroll
                for (int c = 0; c < C; ++c) to[16 * c + l16] = acc[m][c][q];
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
        const bool inside = writes && row < rows && col < p.N;        // (N is a multiple of 8: a thread's columns are in or out together)
        if constexpr (SHARES) {
            static_assert(!SHARES || PER == 1, "64 columns, 16 waves");
            if (inside) p.shares[((int64_t)(blockIdx.z * p.batches + e) * p.M + row) * p.N + col] = v[0];
            continue;
        }
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            v[x] = bf16_to_f32(f32_to_bf16(v[x]));
            if (!GRAD && p.bias && inside) v[x] = bf16_to_f32(f32_to_bf16(v[x] + bf16_to_f32(p.bias[(int64_t)e * p.N + col + x])));
            if (!GRAD && p.relu) v[x] = v[x] < 0.f ? 0.f : v[x];
            if (GRAD && !(inside && bf16_to_f32(p.mask[((int64_t)e * p.M + row) * p.N + col + x]) > 0.f)) v[x] = 0.f;
        }
        if (inside) {
            uint16_t *to = out + (int64_t)row * p.N + col;
            if constexpr (PER == 4) *reinterpret_cast<uint2 *>(to) = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
            else if constexpr (PER == 2) *reinterpret_cast<uint32_t *>(to) = f32x2_to_bf16x2(v[0], v[1]);
            else *to = f32_to_bf16(v[0]);
        }
        if (GRAD && p.colsum) {
            __syncthreads();
#pragma unroll
            for (int x = 0; x < PER; ++x) if (writes) part[row_t * SK_PITCH + col_t + x] = v[x];
            __syncthreads();
            if (tid < SK_COLS)
#pragma unroll
                for (int r = 0; r < 16; ++r) colsum += part[r * SK_PITCH + tid];
        }
    }
    if (GRAD && p.colsum && tid < SK_COLS && n0 + tid < p.N) p.colsum[(int64_t)e * p.N + n0 + tid] = colsum;
}

} // namespace pm
