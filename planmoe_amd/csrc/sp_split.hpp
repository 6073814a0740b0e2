// An fp32 value as the sum of three bf16 values, for products on the bf16 matrix cores (gemm_f32_split.hip).
#pragma once
#include "common.hpp"

namespace pm {

// The matrix cores read subnormal bf16 values as zero.  Times 2^24 every part of every fp32 value is a normal one (the last bit of a
// subnormal fp32 value is 2^-149); what then overflows is found at the end.
constexpr float SP_SCALE = 0x1p24f, SP_UNSCALE = 0x1p-48f;
// two values into their parts, lo in bits 0 .. 15
__device__ __forceinline__ void sp_split(float x0, float x1, uint32_t &h, uint32_t &m, uint32_t &l)
{
    x0 *= SP_SCALE;
    x1 *= SP_SCALE;
    h = f32x2_to_bf16x2(x0, x1);
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
    m = f32x2_to_bf16x2(r0, r1);
    const float s0 = r0 - __uint_as_float(m << 16), s1 = r1 - __uint_as_float(m & 0xffff0000u);
    l = __builtin_amdgcn_perm(__float_as_uint(s1), __float_as_uint(s0), 0x07060302u);
}

} // namespace pm
