// Experts' rows whose product left them in shares (layer_shares.hip).
#pragma once
#include "common.hpp"
#include "gemm_shares.hpp"

namespace pm {

struct RowShares {
    const float *shares;          // [splits][experts * capacity][model_dim]
    int64_t plane;                // floats between shares
    int splits;
    const uint16_t *bias;         // [experts][model_dim], NULL: none
    int capacity, model_dim;
    // eight values of a slot's row, as the product's epilogue would have stored them: the sum rounded, then the bias added in bf16
    __device__ __forceinline__ uint4 vector(int slot, int u) const
    {
        using E = Elem<PLANMOE_BF16>;
        const float4 *src = reinterpret_cast<const float4 *>(shares + (int64_t)slot * model_dim + u * 8);
        float f[8];
        // (four shares at once on their way; the last one again where there are fewer, unused)
        for (int z0 = 0; z0 < splits; z0 += 4) {
            float4 lo[4], hi[4];
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                const float4 *at = src + (int64_t)min(z0 + z, splits - 1) * (plane / 4);
                lo[z] = at[0];
                hi[z] = at[1];
            }
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                const float v[8] = {lo[z].x, lo[z].y, lo[z].z, lo[z].w, hi[z].x, hi[z].y, hi[z].z, hi[z].w};
#pragma unroll
                for (int i = 0; i < 8; ++i) f[i] = z0 + z == 0 ? v[i] : z0 + z < splits ? f[i] + v[i] : f[i];
            }
        }
        uint4 r = E::pack(f);
        if (bias) {
            E::unpack(r, f);
            const uint16_t *b = bias + (int64_t)(slot / capacity) * model_dim + u * 8;
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] += bf16_to_f32(b[i]);
            r = E::pack(f);
        }
        return r;
    }
};

// the combine of such rows through the int8 codec (layer.hip); codes NULL: none are kept
int combine_int8_shares(const char *who, const RowShares &rows, const float *gates, const int32_t *indices, const int32_t *locations, int64_t plane_stride,
                        int top_k, int samples, void *out, uint8_t *codes, void *bias, void *scale, hipStream_t stream);

} // namespace pm
