// The zfp codec (rate 8) on the rows of a layer whose experts' buffers never leave the GPU.
//
// On one rank the all-to-all delivers what was sent, so the codec is decompress(compress(block)) of every 4 slots x 4 columns
// (zfpc.cpp:23-51, 66-86, what overlap.py:12-34 does around a one-rank exchange).  The stream of a block holds its bit planes
// from the top until 128 bits are spent, and what the decoder gives back are those planes: how far they reach follows from their
// lengths alone, so no bits are packed and none are walked, except those of the one plane that the budget ends in.  Blocks of empty
// capacity slots are neither read nor written.
//
// Under the profiler, 4096 x 1024 tokens, top-2, 16 experts x 512 slots: dispatch 16 us, rows in place 17, with their stream kept 21.5, combine's backward
// pass 31, one slot map a pass 9.  (The codec's own entry points, when these kernels took 20, 18, 32, 37 and 10: dispatch with the coder, then
// the decoder 40; coder, then a decoding combine of a launch a choice 16 + 47, where the combine of decoded rows is 9; backward pass 42 + 19; five slot maps 47.)
// Bound by the vector ALUs: 16 bytes a lane and about 600 instructions a block in the dispatch and the rows, the decoder's walk where a stream is read.
#include "zfp_core.hpp"

namespace pm {

constexpr int TRIP_NW = 4;                       // words of a block

// f as the decoder gives it back, same bits; KEEP: the block's stream as well.  A block with an infinity, whose exponent does not fit its
// bits and spills into the first plane's, is coded and decoded.
template <bool KEEP>
__device__ __forceinline__ void zfp_trip16(float (&f)[16], uint32_t *s, const uint16_t *tab)
{
    if (code16<TRIP_NW, KEEP, true>(f, s, tab) != 255) return;
    uint32_t w[TRIP_NW];
    if constexpr (KEEP) {
#pragma unroll
        for (int i = 0; i < TRIP_NW; ++i) w[i] = s[i];
    } else {
        code16<TRIP_NW, true, false>(f, w, group_codes.entry);
    }
    decode16<TRIP_NW>(w, f, walk16_table.step);
}

// slot -> token that fills it, its gate (with `gates`) and its plane; a choice without a slot: its gate gradient is zero.
// Slots in use are those below an expert's count; what the others hold is not used.
__global__ __launch_bounds__(256) void layer_zfp_slots_kernel(const int32_t *__restrict__ indices, const int32_t *__restrict__ locations,
                                                              const float *__restrict__ gates, int64_t stride, int top_k, int samples,
                                                              int experts, int capacity, int32_t *__restrict__ src, float *__restrict__ sgate,
                                                              int32_t *__restrict__ splane, float *__restrict__ grad_gates)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= samples * top_k) return;
    const int j = i / samples, t = i - j * samples;
    const int64_t o = (int64_t)j * stride + t;
    const int e = indices[o], l = locations[o];
    if (e < 0 || e >= experts || l < 0 || l >= capacity) {
        if (grad_gates) grad_gates[o] = 0.f;
        return;
    }
    const int slot = e * capacity + l;
    src[slot] = t;
    if (gates) sgate[slot] = gates[o];
    if (splane) splane[slot] = j;
}

// of the four slots that row of blocks `by` holds, and those behind them, the slots in use
__device__ __forceinline__ int trip_rows_left(int64_t by, const int32_t *counts, int planes, int experts, int capacity)
{
    const int e = (int)((uint32_t)(4 * by) / (uint32_t)capacity);          // (fewer than 2^31 slots)
    int n = 0;
    for (int j = 0; j < planes; ++j) n += counts[j * experts + e];
    return min(n, capacity) - (int)(4 * by - (int64_t)e * capacity);
}
// the block of a thread: row of blocks, column of blocks, how many slots in use there are from its first
struct TripBlock {
    int64_t by;
    int bx, live;
    __device__ __forceinline__ TripBlock(int nbx, int64_t blocks, const int32_t *counts, int planes, int experts, int capacity)
    {
        const int64_t first = (int64_t)blockIdx.x * 256, row = first / nbx;
        const uint32_t at = (uint32_t)(first - row * nbx) + threadIdx.x, down = at / (uint32_t)nbx;
        by = row + down;
        bx = (int)(at - down * (uint32_t)nbx);
        live = first + threadIdx.x < blocks ? trip_rows_left(by, counts, planes, experts, capacity) : 0;
    }
};

// rows[slot] = codec(x[token])
__global__ __launch_bounds__(256) void layer_zfp_dispatch_kernel(const float *__restrict__ x, const int32_t *__restrict__ src,
                                                                 const int32_t *__restrict__ counts, int planes, int samples, int model_dim,
                                                                 int experts, int capacity, int64_t blocks, float *__restrict__ rows)
{
    const TripBlock at(model_dim / 4, blocks, counts, planes, experts, capacity);
    if (at.live <= 0) return;
    const int4 tok = *reinterpret_cast<const int4 *>(src + 4 * at.by);
    const int t[4] = {tok.x, tok.y, tok.z, tok.w};
    float f[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float4 v = *reinterpret_cast<const float4 *>(x + (int64_t)min((uint32_t)t[j], (uint32_t)samples - 1u) * model_dim + 4 * at.bx);
        const bool live = j < at.live;
        f[4 * j] = live ? v.x : 0.f;
        f[4 * j + 1] = live ? v.y : 0.f;
        f[4 * j + 2] = live ? v.z : 0.f;
        f[4 * j + 3] = live ? v.w : 0.f;
    }
    zfp_trip16<false>(f, nullptr, nullptr);
    float *p = rows + 4 * at.by * model_dim + 4 * at.bx;
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<float4 *>(p + (int64_t)j * model_dim) = make_float4(f[4 * j], f[4 * j + 1], f[4 * j + 2], f[4 * j + 3]);
}

// rows = codec(rows) in place; KEEP: their stream as well (a quarter of their size), for the backward pass
template <bool KEEP>
__global__ __launch_bounds__(256) void layer_zfp_rows_kernel(float *__restrict__ rows, const int32_t *__restrict__ counts, int planes,
                                                             int model_dim, int experts, int capacity, int64_t blocks, uint32_t *__restrict__ stream)
{
    __shared__ __align__(4) uint16_t tab[KEEP ? 512 : 2];
    const TripBlock at(model_dim / 4, blocks, counts, planes, experts, capacity);
    if constexpr (KEEP) {
        if (!__syncthreads_or(at.live > 0)) return;
        group_code_table(tab);
    }
    if (at.live <= 0) return;
    float *p = rows + 4 * at.by * model_dim + 4 * at.bx;
    float f[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float4 v = *reinterpret_cast<const float4 *>(p + (int64_t)j * model_dim);
        f[4 * j] = v.x; f[4 * j + 1] = v.y; f[4 * j + 2] = v.z; f[4 * j + 3] = v.w;
    }
    uint32_t w[TRIP_NW];
    zfp_trip16<KEEP>(f, w, tab);
    if constexpr (KEEP) store_words<TRIP_NW>(stream + (at.by * (model_dim / 4) + at.bx) * TRIP_NW, w);
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<float4 *>(p + (int64_t)j * model_dim) = make_float4(f[4 * j], f[4 * j + 1], f[4 * j + 2], f[4 * j + 3]);
}

// Backward of the combine: grad_rows[slot] = codec(gate * grad[token]) and grad_gates = <grad[token], decoded row> from the
// stream that the forward pass kept (GatingDecoder.backward, fast_dispatch.py:62-79).  A work-group owns the four slots of a
// row of blocks; a thread's four partial sums are added in a fixed order.
__global__ __launch_bounds__(256) void layer_zfp_combine_bwd_kernel(const uint32_t *__restrict__ stream, const float *__restrict__ grad,
                                                                    const int32_t *__restrict__ src, const float *__restrict__ sgate,
                                                                    const int32_t *__restrict__ splane, const int32_t *__restrict__ counts,
                                                                    int planes, int64_t stride, int samples, int model_dim, int experts,
                                                                    int capacity, float *__restrict__ grad_rows, float *__restrict__ grad_gates)
{
    __shared__ float s_part[4][4];
    __shared__ __align__(16) uint16_t tab[WALK16_ENTRIES];
    const int64_t by = blockIdx.x;
    const int live = trip_rows_left(by, counts, planes, experts, capacity), nbx = model_dim / 4;
    if (live <= 0) return;                       // (the whole work-group)
    walk16_load(tab);
    const int4 tok = *reinterpret_cast<const int4 *>(src + 4 * by);
    const float4 gv = *reinterpret_cast<const float4 *>(sgate + 4 * by);
    const uint32_t most = (uint32_t)samples - 1u;
    const int64_t t[4] = {min((uint32_t)tok.x, most), min((uint32_t)tok.y, most), min((uint32_t)tok.z, most), min((uint32_t)tok.w, most)};
    const float g[4] = {gv.x, gv.y, gv.z, gv.w};
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int bx = threadIdx.x; bx < nbx; bx += 256) {
        float4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const float4 *>(grad + t[j] * model_dim + 4 * bx);
        uint32_t w[TRIP_NW];
        load_words<TRIP_NW>(stream + (by * nbx + bx) * TRIP_NW, w);
        float f[16];
        decode16<TRIP_NW>(w, f, tab);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc[j] += ((f[4 * j] * v[j].x + f[4 * j + 1] * v[j].y) + f[4 * j + 2] * v[j].z) + f[4 * j + 3] * v[j].w;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f[4 * j] = j < live ? g[j] * v[j].x : 0.f;
            f[4 * j + 1] = j < live ? g[j] * v[j].y : 0.f;
            f[4 * j + 2] = j < live ? g[j] * v[j].z : 0.f;
            f[4 * j + 3] = j < live ? g[j] * v[j].w : 0.f;
        }
        zfp_trip16<false>(f, nullptr, nullptr);
        float *p = grad_rows + 4 * by * model_dim + 4 * bx;
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<float4 *>(p + (int64_t)j * model_dim) = make_float4(f[4 * j], f[4 * j + 1], f[4 * j + 2], f[4 * j + 3]);
    }
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float r = wave_sum(acc[j]);
        if (lane_id() == 0) s_part[wave][j] = r;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        const int j = threadIdx.x;
        if (j < live) {
            const int plane = (int)min((uint32_t)splane[4 * by + j], (uint32_t)planes - 1u);
            grad_gates[(int64_t)plane * stride + min((uint32_t)src[4 * by + j], most)] =
                ((s_part[0][j] + s_part[1][j]) + s_part[2][j]) + s_part[3][j];
        }
    }
}

static int trip_check(const char *who, int model_dim, int experts, int capacity, const int32_t *counts, int planes, int64_t &blocks)
{
    PM_REQUIRE(model_dim >= 1 && experts >= 1 && capacity >= 1 && planes >= 1, "%s: bad shape", who);
    PM_REQUIRE(model_dim % 4 == 0 && capacity % 4 == 0, "%s: model_dim and capacity must be multiples of 4", who);
    PM_REQUIRE((int64_t)experts * capacity < (1ll << 31), "%s: experts*capacity overflows int32", who);
    PM_REQUIRE(counts, "%s: NULL row counts", who);
    blocks = (int64_t)experts * capacity / 4 * (model_dim / 4);
    PM_REQUIRE((blocks + 255) / 256 < (1ll << 31), "%s: too many rows", who);
    return 0;
}

static int trip_planes_check(const char *who, const float *x, const int32_t *indices, const int32_t *locations, int64_t plane_stride, int top_k,
                             int samples, const float *rows, int experts, int capacity, const void *workspace, size_t workspace_bytes)
{
    PM_REQUIRE(x && rows && indices && locations && aligned16(x) && aligned16(rows), "%s: NULL or unaligned argument", who);
    PM_REQUIRE(samples >= 1 && plane_stride >= samples && (int64_t)samples * top_k < (1ll << 31), "%s: bad routing planes", who);
    PM_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= planmoe_layer_zfp_workspace_bytes(experts, capacity), "%s: workspace too small", who);
    return 0;
}

} // namespace pm

using namespace pm;

extern "C" size_t planmoe_layer_zfp_workspace_bytes(int experts, int capacity)
{
    if (experts < 1 || capacity < 1) return 16;
    return (size_t)experts * (size_t)capacity * 12u + 16u;                // slot -> token, gate, plane
}

extern "C" int planmoe_layer_zfp_dispatch(const float *x, const int32_t *indices, const int32_t *locations, int64_t plane_stride,
                                          int top_k, int samples, int model_dim, int experts, int capacity, const int32_t *expert_counts,
                                          float *rows, void *workspace, size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_layer_zfp_dispatch";
    int64_t blocks;
    if (trip_check(who, model_dim, experts, capacity, expert_counts, top_k, blocks) ||
        trip_planes_check(who, x, indices, locations, plane_stride, top_k, samples, rows, experts, capacity, workspace, workspace_bytes)) return 1;
    hipStream_t st = (hipStream_t)stream;
    int32_t *src = (int32_t *)workspace;
    layer_zfp_slots_kernel<<<(unsigned)(((int64_t)samples * top_k + 255) / 256), 256, 0, st>>>(
        indices, locations, nullptr, plane_stride, top_k, samples, experts, capacity, src, nullptr, nullptr, nullptr);
    layer_zfp_dispatch_kernel<<<(unsigned)((blocks + 255) / 256), 256, 0, st>>>(x, src, expert_counts, top_k, samples, model_dim, experts, capacity,
                                                                                blocks, rows);
    PM_LAUNCH_CHECK(who);
    return 0;
}

extern "C" int planmoe_layer_zfp_rows(float *rows, int model_dim, int experts, int capacity, const int32_t *expert_counts, int planes,
                                      void *stream_out, size_t stream_capacity, void *stream)
{
    const char *who = "planmoe_layer_zfp_rows";
    int64_t blocks;
    if (trip_check(who, model_dim, experts, capacity, expert_counts, planes, blocks)) return 1;
    PM_REQUIRE(rows && aligned16(rows) && aligned16(stream_out), "%s: NULL or unaligned argument", who);
    PM_REQUIRE(!stream_out || stream_capacity >= (size_t)blocks * TRIP_NW * 4, "%s: stream buffer too small", who);
    hipStream_t st = (hipStream_t)stream;
    const unsigned grid = (unsigned)((blocks + 255) / 256);
    if (stream_out) layer_zfp_rows_kernel<true><<<grid, 256, 0, st>>>(rows, expert_counts, planes, model_dim, experts, capacity, blocks, (uint32_t *)stream_out);
    else layer_zfp_rows_kernel<false><<<grid, 256, 0, st>>>(rows, expert_counts, planes, model_dim, experts, capacity, blocks, nullptr);
    PM_LAUNCH_CHECK(who);
    return 0;
}

extern "C" int planmoe_layer_zfp_combine_bwd(const void *stream_in, const float *grad, const float *gates, const int32_t *indices,
                                             const int32_t *locations, int64_t plane_stride, int top_k, int samples, int model_dim,
                                             int experts, int capacity, const int32_t *expert_counts, float *grad_rows, float *grad_gates,
                                             void *workspace, size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_layer_zfp_combine_bwd";
    int64_t blocks;
    if (trip_check(who, model_dim, experts, capacity, expert_counts, top_k, blocks) ||
        trip_planes_check(who, grad, indices, locations, plane_stride, top_k, samples, grad_rows, experts, capacity, workspace, workspace_bytes)) return 1;
    PM_REQUIRE(stream_in && aligned16(stream_in) && gates && grad_gates, "%s: NULL argument", who);
    hipStream_t st = (hipStream_t)stream;
    const int64_t slots = (int64_t)experts * capacity;
    int32_t *src = (int32_t *)workspace, *splane = src + 2 * slots;
    float *sgate = (float *)(src + slots);
    layer_zfp_slots_kernel<<<(unsigned)(((int64_t)samples * top_k + 255) / 256), 256, 0, st>>>(
        indices, locations, gates, plane_stride, top_k, samples, experts, capacity, src, sgate, splane, grad_gates);
    layer_zfp_combine_bwd_kernel<<<(unsigned)(slots / 4), 256, 0, st>>>((const uint32_t *)stream_in, grad, src, sgate, splane, expert_counts, top_k,
                                                                        plane_stride, samples, model_dim, experts, capacity, grad_rows, grad_gates);
    PM_LAUNCH_CHECK(who);
    return 0;
}
