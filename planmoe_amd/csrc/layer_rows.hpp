// The "int8" codec of a row that a wave holds in registers, as the layer's row passes apply it.
#pragma once
#include "rows.hpp"
#include "int8_core.hpp"

namespace pm {

// a vector's codes as they are kept, one byte a value
template <int DT> struct CodeWords { uint32_t w[Elem<DT>::VEC / 4]; };
template <int DT>
__device__ __forceinline__ void store_codes(uint8_t *to, const CodeWords<DT> &v)
{
    if constexpr (Elem<DT>::VEC == 8) stream_store(reinterpret_cast<uint2 *>(to), make_uint2(v.w[0], v.w[1]));
    else stream_store(reinterpret_cast<uint32_t *>(to), v.w[0]);
}

// decompress(compress(row)) of a row held as CACHE vectors per lane (vectors past the end: copies of the last);
// keep(c, codes) sees the codes of vector c.  Returns the row's minimum and scale.
template <int DT, int CACHE, bool CANON, typename Keep>
__device__ __forceinline__ float2 through_int8(uint4 (&row)[CACHE], Keep keep)
{
    using E = Elem<DT>;
    RowStats<DT, CANON> stats;
    stats.init();
#pragma unroll
    for (int c = 0; c < CACHE; ++c) stats.add(row[c]);
    float mn, mx;
    stats.finish(mn, mx);
    const float scale = E::round(mx - mn);
    const RowEncoder<DT> enc(mn, scale);
    const RowDecoder<DT> dec(mn, scale);
    auto body = [&](auto mode) {
#pragma unroll
        for (int c = 0; c < CACHE; ++c) {
            CodeWords<DT> code;
            float f[E::VEC];
            enc.template encode<decltype(mode)::value>(row[c], code.w);
            keep(c, code);
#pragma unroll
            for (int q = 0; q < E::VEC / 4; ++q) dec.word(code.w[q], f + 4 * q);
            row[c] = E::pack(f);
        }
    };
    if (enc.fast()) body(std::true_type{}); else body(std::false_type{});
    return make_float2(mn, scale);
}

// The same with the decoder as a table: a row has 256 codes, so a wave works out gate * decoded(code) for four codes a
// lane, into LDS, and a value is a lookup by its code.  (Decoding value by value, the 35 vector instructions of a pair
// of bf16 values took as long as its bytes.  Combine at 16384 x 4096, top-2, 113 -> 81 us,
// at 16384 x 1024 35 -> 27, its backward pass there 64 -> 48.)
template <int DT>
__device__ __forceinline__ void fill_table(float mn, float scale, float gate, float *table)
{
    float f[4];
    RowDecoder<DT>(mn, scale).word(0x03020100u + 0x04040404u * (uint32_t)lane_id(), f);
    *reinterpret_cast<float4 *>(table + 4 * lane_id()) = make_float4(gate * f[0], gate * f[1], gate * f[2], gate * f[3]);
}
template <int DT>
struct RowTable {
    RowEncoder<DT> enc;
    const float *tab;                            // 256 values, the wave's own
    float mn, scale;
    template <int CACHE>
    __device__ __forceinline__ RowTable(const uint4 (&row)[CACHE], float gate, float *table) : enc(0.f, 0.f), tab(table)
    {
        using E = Elem<DT>;
        RowStats<DT, false> stats;
        stats.init();
#pragma unroll
        for (int c = 0; c < CACHE; ++c) stats.add(row[c]);
        float mx;
        stats.finish(mn, mx);
        scale = E::round(mx - mn);
        enc = RowEncoder<DT>(mn, scale);
        fill_table<DT>(mn, scale, gate, table);
    }
    template <bool FAST, typename Keep>
    __device__ __forceinline__ void values(const uint4 &raw, float (&f)[Elem<DT>::VEC], Keep keep) const
    {
        uint32_t c[Elem<DT>::VEC];
        enc.template codes<FAST>(raw, c);
        CodeWords<DT> code;
#pragma unroll
        for (int q = 0; q < Elem<DT>::VEC / 4; ++q) code.w[q] = c[4 * q] | (c[4 * q + 1] << 8) | (c[4 * q + 2] << 16) | (c[4 * q + 3] << 24);
        keep(code);
#pragma unroll
        for (int i = 0; i < Elem<DT>::VEC; ++i) f[i] = tab[c[i]];
    }
    template <bool FAST>
    __device__ __forceinline__ void values(const uint4 &raw, float (&f)[Elem<DT>::VEC]) const
    {
        values<FAST>(raw, f, [](const CodeWords<DT> &) {});
    }
};
// what a wave's lanes wrote to its LDS is there for all of them, and what they read has been read
__device__ __forceinline__ void table_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the rows a wave keeps in registers: 1, 2, 4, 8 or 16 vectors per lane
#define PM_ROW_CACHE(CALL)                                    \
    do {                                                      \
        if (per_lane <= 1) CALL(1);                           \
        else if (per_lane <= 2) CALL(2);                      \
        else if (per_lane <= 4) CALL(4);                      \
        else if (per_lane <= 8) CALL(8);                      \
        else CALL(16);                                        \
    } while (0)

// what the layer's row passes ask of their arguments
int layer_rows_check(const char *who, int dtype, const void *rows, const int32_t *indices, const int32_t *locations, int64_t stride,
                     int top_k, int samples, int model_dim, int experts, int capacity, int codec);

} // namespace pm
