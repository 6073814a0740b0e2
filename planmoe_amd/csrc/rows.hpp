// Row access helpers shared by the kernels that move token rows to and from capacity slots.
#pragma once
#include "common.hpp"
#include <type_traits>

namespace pm {

// How a lane reaches a row's elements.  ROWS_16: rows of 16-byte vectors, 16-byte aligned.  ROWS_4: rows of whole
// dwords, at least one vector long, as 16-byte accesses that are dword aligned, the last one moved back to end with
// the row (its first elements are the ones the vector before it holds; stored twice with the same
// value).  ROWS_1: element by element (3001 x 1030 fp16, three choices, dispatch: 13.8 us, 6.5 as ROWS_4).
enum { ROWS_1 = 0, ROWS_4 = 1, ROWS_16 = 2 };

typedef uint32_t pm_u32x4_dwords __attribute__((ext_vector_type(4), aligned(4)));

template <int DT, int MODE, bool STREAM = true>
struct RowIO {
    using E = Elem<DT>;
    static constexpr int U = MODE ? E::VEC : 1;        // elements per lane access
    static constexpr int BYTES = U * (int)sizeof(typename E::store_t);
    __host__ __device__ static __forceinline__ int units(int model_dim) { return (model_dim + U - 1) / U; }
    // byte offset of unit u in a row of `bytes`
    __device__ static __forceinline__ int at(int u, int bytes) { return MODE == ROWS_4 ? min(u * BYTES, bytes - BYTES) : u * BYTES; }
    __device__ static __forceinline__ void load(const void *row, int off, float *f)
    {
        const char *p = (const char *)row + off;
        if constexpr (MODE == ROWS_16) {
            E::unpack(*reinterpret_cast<const uint4 *>(p), f);
        } else if constexpr (MODE == ROWS_4) {
            const pm_u32x4_dwords v = *reinterpret_cast<const pm_u32x4_dwords *>(p);
            E::unpack(make_uint4(v.x, v.y, v.z, v.w), f);
        } else {
            f[0] = E::load(p, 0);
        }
    }
    // what a lane has asked for, kept as it lies in memory until it is used
    typedef std::conditional_t<MODE == ROWS_1, float, uint4> raw_t;
    __device__ static __forceinline__ raw_t load_raw(const void *row, int off)
    {
        const char *p = (const char *)row + off;
        if constexpr (MODE == ROWS_16) {
            return *reinterpret_cast<const uint4 *>(p);
        } else if constexpr (MODE == ROWS_4) {
            const pm_u32x4_dwords v = *reinterpret_cast<const pm_u32x4_dwords *>(p);
            return make_uint4(v.x, v.y, v.z, v.w);
        } else {
            return E::load(p, 0);
        }
    }
    __device__ static __forceinline__ void unpack(const raw_t &v, float *f)
    {
        if constexpr (MODE == ROWS_1) f[0] = v;
        else E::unpack(v, f);
    }
    // for launches that store nothing in bulk (measured: streaming loads next to streaming
    // stores slow the dispatch / combine kernels down, alone they help)
    __device__ static __forceinline__ void load_stream(const void *row, int off, float *f)
    {
        const char *p = (const char *)row + off;
        if constexpr (MODE == ROWS_16) {
            E::unpack(stream_load(reinterpret_cast<const uint4 *>(p)), f);
        } else if constexpr (MODE == ROWS_4) {
            const pm_u32x4_dwords v = __builtin_nontemporal_load(reinterpret_cast<const pm_u32x4_dwords *>(p));
            E::unpack(make_uint4(v.x, v.y, v.z, v.w), f);
        } else {
            f[0] = E::load(p, 0);
        }
    }
    __device__ static __forceinline__ void store_bits(void *row, int off, const uint4 &v)
    {
        char *p = (char *)row + off;
        if constexpr (MODE == ROWS_16 && STREAM) stream_store(reinterpret_cast<uint4 *>(p), v);
        else if constexpr (MODE == ROWS_16) *reinterpret_cast<uint4 *>(p) = v;
        else *reinterpret_cast<pm_u32x4_dwords *>(p) = pm_u32x4_dwords{v.x, v.y, v.z, v.w};
    }
    __device__ static __forceinline__ void store(void *row, int off, const float *f)
    {
        if constexpr (MODE != ROWS_1) store_bits(row, off, E::pack(f));
        else E::store((char *)row + off, 0, f[0]);
    }
    __device__ static __forceinline__ void store_zero(void *row, int off)
    {
        if constexpr (MODE != ROWS_1) store_bits(row, off, make_uint4(0, 0, 0, 0));
        else E::store((char *)row + off, 0, 0.f);
    }
};

inline int rows_mode(int dtype, int model_dim, const void *a, const void *b)
{
    const int vec = dtype == PLANMOE_F32 ? 4 : 8, size = dtype == PLANMOE_F32 ? 4 : 2;
    if (model_dim % vec == 0 && aligned16(a) && aligned16(b)) return ROWS_16;
    const bool dwords = ((uintptr_t)a | (uintptr_t)b) % 4 == 0 && model_dim * size % 4 == 0;
    return dwords && model_dim >= vec ? ROWS_4 : ROWS_1;
}
#define PM_ROWS_SWITCH(mode, MODE, ...)                                                  \
    do {                                                                                 \
        if ((mode) == ROWS_16) { constexpr int MODE = ROWS_16; __VA_ARGS__; }            \
        else if ((mode) == ROWS_4) { constexpr int MODE = ROWS_4; __VA_ARGS__; }         \
        else { constexpr int MODE = ROWS_1; __VA_ARGS__; }                               \
    } while (0)

__device__ __forceinline__ int   rl_i(int v, int lane)   { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float rl_f(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }

// Lane j (< nplanes) of the calling wave fetches plane j0+j of token t: its slot row
// (-1 when the pair is not live) and its gate.
__device__ __forceinline__ void fetch_planes(const float *gates, const int32_t *indices,
                                             const int32_t *locations, int64_t stride, int t,
                                             int j0, int nplanes, int experts, int capacity,
                                             int &slot, float &gate)
{
    slot = -1; gate = 1.f;
    const int lane = lane_id();
    if (lane < nplanes) {
        const int64_t o = (int64_t)(j0 + lane) * stride + t;
        const int e = indices[o], l = locations[o];
        if (e >= 0 && e < experts && l >= 0 && l < capacity) slot = e * capacity + l;
        if (gates) gate = gates[o];
    }
}

// Which slots no live pair addresses.  Up to SLOT_FILL_PAIRS pairs (of narrow rows fewer: slot_fill) the work-groups that write those slots' zero
// rows find out themselves: there are 2^shift of them, one in 2^shift slots is a work-group's, and it walks the routing planes, 16 loads at once, and
// keeps a bit a slot in LDS.  They are the first of the grid, so that the walk is beside the rows of the tokens.  (Two small launches in front for
// flags in memory cost 9 us of 193 in the routing API's pass at 8192 x 2048, and 10 us of host time in any.)  More pairs: flags.
constexpr int SLOT_FILL_PAIRS = 1 << 17, SLOT_FILL_BITS = 8192;
struct SlotFill {
    const uint32_t *flags;                       // NULL: bits in LDS
    int blocks, shift;                           // work-groups that fill
    // work-group b of the grid: below zero its number among those that fill is ~b, else its number among those of the tokens
    __device__ __forceinline__ int role(int b, int token_blocks) const
    {
        if (flags) return b >= token_blocks ? ~(b - token_blocks) : b;
        return b < blocks ? ~b : b - blocks;
    }
};
// zero(slot) for every empty slot of work-group `number`, a wave each
template <typename Zero>
__device__ __forceinline__ void fill_empty_slots(const SlotFill &fill, int number, const int32_t *__restrict__ indices,
                                                 const int32_t *__restrict__ locations, int64_t stride, int top_k, int samples, int experts,
                                                 int capacity, Zero zero)
{
    const int wave = threadIdx.x >> 6, slots = experts * capacity;
    if (fill.flags) {
        for (int s = number * 4 + wave; s < slots; s += fill.blocks * 4)
            if (!fill.flags[s]) zero(s);
        return;
    }
    __shared__ uint32_t s_used[SLOT_FILL_BITS / 32];
    constexpr int AT_ONCE = 16;
    const int mine = (slots - number + (1 << fill.shift) - 1) >> fill.shift;          // slots number, number + 2^shift, ..
    for (int i = threadIdx.x; i < (mine + 31) / 32; i += 256) s_used[i] = 0u;
    __syncthreads();
    for (int j = 0; j < top_k; ++j) {
        const int32_t *idx = indices + (int64_t)j * stride, *loc = locations + (int64_t)j * stride;
        for (int t0 = threadIdx.x; t0 < samples; t0 += AT_ONCE * 256) {
            int e[AT_ONCE], l[AT_ONCE];
#pragma unroll
            for (int q = 0; q < AT_ONCE; ++q) {
                const int t = min(t0 + q * 256, samples - 1);      // (the last token again and again: its bit is its own)
                e[q] = idx[t];
                l[q] = loc[t];
            }
#pragma unroll
            for (int q = 0; q < AT_ONCE; ++q) {
                const int s = e[q] * capacity + l[q], at = s >> fill.shift;
                if (e[q] >= 0 && e[q] < experts && l[q] >= 0 && l[q] < capacity && (s & ((1 << fill.shift) - 1)) == number) atomicOr(&s_used[at >> 5], 1u << (at & 31));
            }
        }
    }
    __syncthreads();
    for (int i = wave; i < mine; i += 4)
        if (!((s_used[i >> 5] >> (i & 31)) & 1u)) zero(number + (i << fill.shift));
}
// how the empty slots are found: the flags' launches, or nothing beforehand
SlotFill slot_fill(void *workspace, const int32_t *indices, const int32_t *locations, int64_t stride, int top_k, int samples, int experts,
                   int capacity, int64_t row_bytes, hipStream_t st);
int check_planes(const char *who, const int32_t *indices, const int32_t *locations,
                 int64_t stride, int top_k, int samples);
// routing of up to 64 experts from [samples, experts] logits / scores with the forward chain's
// epilogue; workspace of planmoe_forward_workspace_bytes(samples, experts, top_k)
int route_groups(const void *input, int dtype, int is_logits, const float *logit_bias, int samples, int experts,
                 int top_k, int normalize_gate, int32_t *indices, int32_t *locations, void *gates, int64_t stride,
                 void *scores_out, float *l_aux, int32_t *counts, void *workspace, hipStream_t st);

} // namespace pm
