// Dispatch / combine / gate-gradient kernels: the token <-> capacity-slot row movers.
//
// They take the place of the three JIT-compiled CUDA kernels of the reference
// (jit_kernels/sparse.py:17-134) and of the per-choice launch loops around them
// (impls/fast_dispatch.py:16-79).  Layout: x / out are [samples, model_dim] rows,
// dispatched is [experts * capacity, model_dim] rows; one wavefront owns one token row and
// moves it with 16-byte accesses, all k choices of the token in the same pass.
#include "rows.hpp"

#include <algorithm>

namespace pm {

// ------------------------------------------------------------------ slot occupancy flags
__global__ __launch_bounds__(256) void slot_flags_clear(uint32_t *flags, int slots)
{
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < slots) flags[i] = 0u;
}

__global__ __launch_bounds__(256) void slot_flags_mark(uint32_t *flags, const int32_t *indices,
                                                       const int32_t *locations, int64_t stride,
                                                       int top_k, int samples, int experts,
                                                       int capacity)
{
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= samples * top_k) return;
    int j = i / samples, t = i - j * samples;
    int64_t o = (int64_t)j * stride + t;
    int e = indices[o], l = locations[o];
    if (e >= 0 && e < experts && l >= 0 && l < capacity) flags[e * capacity + l] = 1u;
}

// ------------------------------------------------------------------ dispatch (scatter rows)
// token_blocks work-groups move token rows: dispatched[slot] = 0 + gate * x[t]; the others write zero rows into the slots
// no live pair addresses.  Bound by memory: 8192 x 2048 fp32, two choices, 201 MB in 31 us, 14020 x 3528 bf16 317 MB in 69 (a unit at a
// time 32 and 77).
template <int DT, int MODE, bool STREAM>
__global__ __launch_bounds__(256) void dispatch_kernel(
    const void *__restrict__ x, const float *__restrict__ gates,
    const int32_t *__restrict__ indices, const int32_t *__restrict__ locations, int64_t stride,
    int top_k, int samples, int model_dim, int experts, int capacity,
    void *__restrict__ dispatched, const SlotFill fill, int token_blocks)
{
    using IO = RowIO<DT, MODE, STREAM>;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int units = IO::units(model_dim);
    const int64_t row_bytes = (int64_t)model_dim * sizeof(typename Elem<DT>::store_t);

    const int number = fill.role((int)blockIdx.x, token_blocks);
    if (number < 0) {
        fill_empty_slots(fill, ~number, indices, locations, stride, top_k, samples, experts, capacity, [&](int s) {
            char *row = (char *)dispatched + (int64_t)s * row_bytes;
            for (int u = lane; u < units; u += WAVE) IO::store_zero(row, IO::at(u, (int)row_bytes));
        });
        return;
    }

    const int t = number * 4 + wave;
    if (t >= samples) return;
    const char *src = (const char *)x + (int64_t)t * row_bytes;

    for (int j0 = 0; j0 < top_k; j0 += WAVE) {
        const int np = min(top_k - j0, WAVE);
        int slot; float gate;
        fetch_planes(gates, indices, locations, stride, t, j0, np, experts, capacity, slot, gate);
        if (__ballot(slot >= 0) == 0) continue;          // every choice of this pass dropped: the row is not read
        // four units of a row per lane are asked for before the first is stored: a wait for a load waits for the stores
        // ahead of it too, and there is one a unit where they alternate
        constexpr int B = 4;
        for (int u0 = lane; u0 < units; u0 += B * WAVE) {
            typename IO::raw_t row[B];
#pragma unroll
            for (int b = 0; b < B; ++b) row[b] = IO::load_raw(src, IO::at(min(u0 + b * WAVE, units - 1), (int)row_bytes));
            for (int j = 0; j < np; ++j) {
                const int s = rl_i(slot, j);
                if (s < 0) continue;
                const float g = rl_f(gate, j);
                char *to = (char *)dispatched + (int64_t)s * row_bytes;
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    float v[IO::U], o[IO::U];
                    IO::unpack(row[b], v);
#pragma unroll
                    for (int i = 0; i < IO::U; ++i) o[i] = 0.f + g * v[i];
                    if (u0 + b * WAVE < units) IO::store(to, IO::at(u0 + b * WAVE, (int)row_bytes), o);
                }
            }
        }
    }
}

// ------------------------------------------------------------------ combine (gather rows)
// out[t] = sum_j (live_j ? gate_j * dispatched[slot_j] : 0), planes added left to right.  Bound by memory.  A wave asks for B units a lane
// of two choices' rows before it adds any (a dropped choice reads slot 0 and contributes zeros): one wait a pass over 4 KB rows, and
// over 8 KB rows with B = 8 (8192 x 2048 fp32, two choices, 201 MB: 36.7 us, 38.5 with four units of one choice at a time, 38.8 of two; 14020 x 3528 bf16
// 54.8, 57.7, 57.5; rows of 2 KB lose with eight: 16384 x 1024 bf16 17.5 and 23.6; which rows take one and which eight: planmoe_combine_fwd).
template <int DT, int MODE, int B>
__global__ __launch_bounds__(256) void combine_kernel(
    const void *__restrict__ dispatched, const float *__restrict__ gates,
    const int32_t *__restrict__ indices, const int32_t *__restrict__ locations, int64_t stride,
    int top_k, int samples, int model_dim, int capacity, void *__restrict__ out)
{
    using IO = RowIO<DT, MODE>;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int units = IO::units(model_dim);
    const int64_t row_bytes = (int64_t)model_dim * sizeof(typename Elem<DT>::store_t);
    const int t = blockIdx.x * 4 + wave;
    if (t >= samples) return;
    char *dst = (char *)out + (int64_t)t * row_bytes;

    if (top_k <= WAVE) {
        int slot; float gate;
        fetch_planes(gates, indices, locations, stride, t, 0, top_k, 0x7fffffff, capacity, slot, gate);
        for (int u0 = lane; u0 < units; u0 += B * WAVE) {
            float acc[B][IO::U];
            constexpr int G = 2;
            for (int j0 = 0; j0 < top_k; j0 += G) {
                typename IO::raw_t row[G][B];
#pragma unroll
                for (int j = 0; j < G; ++j) {
                    if (j0 + j >= top_k) break;
                    const char *from = (const char *)dispatched + (int64_t)max(rl_i(slot, j0 + j), 0) * row_bytes;
#pragma unroll
                    for (int b = 0; b < B; ++b) row[j][b] = IO::load_raw(from, IO::at(min(u0 + b * WAVE, units - 1), (int)row_bytes));
                }
#pragma unroll
                for (int j = 0; j < G; ++j) {
                    if (j0 + j >= top_k) break;
                    const int s = rl_i(slot, j0 + j);
                    const float g = rl_f(gate, j0 + j);
#pragma unroll
                    for (int b = 0; b < B; ++b) {
                        float term[IO::U];
                        IO::unpack(row[j][b], term);
#pragma unroll
                        for (int i = 0; i < IO::U; ++i) {
                            const float v = s >= 0 ? g * term[i] : 0.f;
                            acc[b][i] = (j0 + j == 0) ? v : acc[b][i] + v;
                        }
                    }
                }
            }
#pragma unroll
            for (int b = 0; b < B; ++b)
                if (u0 + b * WAVE < units) IO::store(dst, IO::at(u0 + b * WAVE, (int)row_bytes), acc[b]);
        }
    } else {
        // more planes than lanes: walk the planes straight from memory
        for (int u = lane; u < units; u += WAVE) {
            float acc[IO::U];
            for (int j = 0; j < top_k; ++j) {
                const int64_t o = (int64_t)j * stride + t;
                const int e = indices[o], l = locations[o];
                const float g = gates ? gates[o] : 1.f;
                float term[IO::U];
                if (e >= 0 && l >= 0 && l < capacity) {
                    IO::load((const char *)dispatched + ((int64_t)e * capacity + l) * row_bytes, IO::at(u, (int)row_bytes), term);
#pragma unroll
                    for (int i = 0; i < IO::U; ++i) term[i] = g * term[i];
                } else {
#pragma unroll
                    for (int i = 0; i < IO::U; ++i) term[i] = 0.f;
                }
#pragma unroll
                for (int i = 0; i < IO::U; ++i) acc[i] = (j == 0) ? term[i] : acc[i] + term[i];
            }
            IO::store(dst, IO::at(u, (int)row_bytes), acc);
        }
    }
}

template <int DT, int MODE>
__global__ __launch_bounds__(256) void zero_rows_kernel(void *__restrict__ out, int samples, int model_dim)
{
    using IO = RowIO<DT, MODE>;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= samples) return;
    const int row_bytes = model_dim * (int)sizeof(typename Elem<DT>::store_t);
    char *dst = (char *)out + (int64_t)t * row_bytes;
    for (int u = lane_id(); u < IO::units(model_dim); u += WAVE) IO::store_zero(dst, IO::at(u, row_bytes));
}

// ------------------------------------------------------------------ gate gradient
// grad_gates[j][t] = <dispatched[slot_j], x[t]> (0 for a dropped pair).  One wave per token;
// planes are taken four at a time so the token row is read once per group.  Rows that are not 16-byte aligned go
// element by element, also where they could be read as dwords: where a token's choices hold the same row, what
// the normalised gates pass on is the rounding of these sums alone, and their order stays what it is.
template <int DT, int MODE>
__global__ __launch_bounds__(256) void bwd_gate_kernel(
    const void *__restrict__ x, const void *__restrict__ dispatched,
    const int32_t *__restrict__ indices, const int32_t *__restrict__ locations, int64_t stride,
    int top_k, int samples, int model_dim, int capacity, float *__restrict__ grad_gates)
{
    using IO = RowIO<DT, MODE>;
    constexpr int G = 4;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int units = IO::units(model_dim);
    const int64_t row_bytes = (int64_t)model_dim * sizeof(typename Elem<DT>::store_t);
    const int t = blockIdx.x * 4 + wave;
    if (t >= samples) return;
    const char *xr = (const char *)x + (int64_t)t * row_bytes;

    for (int j0 = 0; j0 < top_k; j0 += G) {
        const int np = min(G, top_k - j0);
        int slot; float gate;
        fetch_planes(nullptr, indices, locations, stride, t, j0, np, 0x7fffffff, capacity, slot, gate);
        int s[G];
#pragma unroll
        for (int j = 0; j < G; ++j) s[j] = (j < np) ? rl_i(slot, j) : -1;
        float acc[G] = {0.f, 0.f, 0.f, 0.f};
        // two vectors or eight elements of the row per lane and pass; the slot rows of all choices are requested with
        // straight-line loads at clamped addresses (a dropped choice reads slot 0 and is left out
        // of the sum; the caller guarantees a slot 0 to read: capacity >= 1)
        constexpr int B = MODE == ROWS_16 ? 2 : 8;
        for (int u0 = lane; u0 < units; u0 += B * WAVE) {
            float a[B][IO::U];
#pragma unroll
            for (int b = 0; b < B; ++b) IO::load_stream(xr, IO::at(min(u0 + b * WAVE, units - 1), (int)row_bytes), a[b]);
#pragma unroll
            for (int j = 0; j < G; ++j) {
                if (j < np) {
                    const char *row = (const char *)dispatched + (int64_t)max(s[j], 0) * row_bytes;
                    float d[B][IO::U];
#pragma unroll
                    for (int b = 0; b < B; ++b) IO::load_stream(row, IO::at(min(u0 + b * WAVE, units - 1), (int)row_bytes), d[b]);
#pragma unroll
                    for (int b = 0; b < B; ++b) {
                        const bool live = s[j] >= 0 && u0 + b * WAVE < units;
#pragma unroll
                        for (int i = 0; i < IO::U; ++i) acc[j] = live ? fmaf(d[b][i], a[b][i], acc[j]) : acc[j];
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < G; ++j) {
            if (j >= np) break;
            const float r = wave_sum(acc[j]);
            if (lane == 0) grad_gates[(int64_t)(j0 + j) * stride + t] = r;
        }
    }
}

// ------------------------------------------------------------------ combine's backward pass
// dispatch_kernel's scatter of the gated gradient and bwd_gate_kernel's products in one pass over the gradient:
// grad_rows[slot_j] = 0 + gate_j * grad[t], grad_gates[j][t] = <rows[slot_j], grad[t]>.  Bound by memory (8192 x
// 2048 fp32, two choices: 335 MB where the two launches move 402).
template <int DT, int MODE, bool STREAM>
__global__ __launch_bounds__(256) void combine_bwd_kernel(
    const void *__restrict__ grad, const void *__restrict__ rows, const float *__restrict__ gates,
    const int32_t *__restrict__ indices, const int32_t *__restrict__ locations, int64_t stride,
    int top_k, int samples, int model_dim, int experts, int capacity,
    void *__restrict__ grad_rows, float *__restrict__ grad_gates, const SlotFill fill, int token_blocks)
{
    using IO = RowIO<DT, MODE, STREAM>;
    constexpr int G = 4, B = 2;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int units = IO::units(model_dim);
    const int row_bytes = model_dim * (int)sizeof(typename Elem<DT>::store_t);

    const int number = fill.role((int)blockIdx.x, token_blocks);
    if (number < 0) {
        fill_empty_slots(fill, ~number, indices, locations, stride, top_k, samples, experts, capacity, [&](int s) {
            char *row = (char *)grad_rows + (int64_t)s * row_bytes;
            for (int u = lane; u < units; u += WAVE) IO::store_zero(row, IO::at(u, row_bytes));
        });
        return;
    }

    const int t = number * 4 + wave;
    if (t >= samples) return;
    const char *gr = (const char *)grad + (int64_t)t * row_bytes;
    for (int j0 = 0; j0 < top_k; j0 += G) {
        const int np = min(G, top_k - j0);
        int slot; float gate;
        fetch_planes(gates, indices, locations, stride, t, j0, np, experts, capacity, slot, gate);
        int s[G];
        float g[G], acc[G];
#pragma unroll
        for (int j = 0; j < G; ++j) { s[j] = j < np ? rl_i(slot, j) : -1; g[j] = rl_f(gate, j); acc[j] = 0.f; }
        if constexpr (MODE == ROWS_16) {
            for (int u0 = lane; u0 < units; u0 += B * WAVE) {
                int off[B];
                float a[B][IO::U];
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    off[b] = IO::at(min(u0 + b * WAVE, units - 1), row_bytes);
                    IO::load(gr, off[b], a[b]);
                }
                // every choice's row is requested before the first is used (a dropped choice reads slot 0, unused: capacity >= 1)
                float d[G][B][IO::U];
#pragma unroll
                for (int j = 0; j < G; ++j)
                    if (j < np) {
#pragma unroll
                        for (int b = 0; b < B; ++b) IO::load((const char *)rows + (int64_t)max(s[j], 0) * row_bytes, off[b], d[j][b]);
                    }
#pragma unroll
                for (int j = 0; j < G; ++j) {
                    if (s[j] < 0) continue;
                    char *to = (char *)grad_rows + (int64_t)s[j] * row_bytes;
#pragma unroll
                    for (int b = 0; b < B; ++b) {
                        const bool live = u0 + b * WAVE < units;
                        float o[IO::U];
#pragma unroll
                        for (int i = 0; i < IO::U; ++i) {
                            acc[j] = live ? fmaf(d[j][b][i], a[b][i], acc[j]) : acc[j];
                            o[i] = 0.f + g[j] * a[b][i];
                        }
                        if (live) IO::store(to, off[b], o);
                    }
                }
            }
        } else {
            // rows as dwords for the scatter, then (from the caches) element by element for the sums, as bwd_gate_kernel
            for (int u = lane; u < units; u += WAVE) {
                const int off = IO::at(u, row_bytes);
                float a[IO::U];
                IO::load(gr, off, a);
#pragma unroll
                for (int j = 0; j < G; ++j) {
                    if (s[j] < 0) continue;
                    float o[IO::U];
#pragma unroll
                    for (int i = 0; i < IO::U; ++i) o[i] = 0.f + g[j] * a[i];
                    IO::store((char *)grad_rows + (int64_t)s[j] * row_bytes, off, o);
                }
            }
            using E = Elem<DT>;
            constexpr int S = 8;
            for (int u0 = lane; u0 < model_dim; u0 += S * WAVE) {
                float a[S], d[G][S];
#pragma unroll
                for (int b = 0; b < S; ++b) a[b] = E::load(gr, min(u0 + b * WAVE, model_dim - 1));
#pragma unroll
                for (int j = 0; j < G; ++j)
                    if (j < np) {
#pragma unroll
                        for (int b = 0; b < S; ++b)
                            d[j][b] = E::load((const char *)rows + (int64_t)max(s[j], 0) * row_bytes, min(u0 + b * WAVE, model_dim - 1));
                    }
#pragma unroll
                for (int j = 0; j < G; ++j)
#pragma unroll
                    for (int b = 0; b < S; ++b) acc[j] = s[j] >= 0 && u0 + b * WAVE < model_dim ? fmaf(d[j][b], a[b], acc[j]) : acc[j];
            }
        }
#pragma unroll
        for (int j = 0; j < G; ++j) {
            if (j >= np) break;
            const float r = wave_sum(acc[j]);
            if (lane == 0) grad_gates[(int64_t)(j0 + j) * stride + t] = r;
        }
    }
}

// Rows that the call after this one reads are stored past the caches where they would not all be there by then, and plainly where the 256 MB of
// the memory-side cache hold them: what follows a dispatch reads its rows, a combine's backward pass reads rows and writes as many.  us, dispatch, combine, its
// backward pass, combine, by what is stored plainly: none, the dispatch's rows, the backward pass's too
//   rows of 134 MB in all 174, 162, 159     218 MB 281, 267, 284     246 MB 270, 262, 274     335 MB 374, 399, 420     84 MB 104.6, 101.9, 99.2
// (What a combine stores is stored past them: 8192 x 2048 fp32 171 in place of 159.)  A call alone, one after the other into the same rows that nothing reads, is up to 16 % slower for
// it (5779 x 2176 fp16 dispatch 13.5 and 15.7), with the combine behind it 500 sizes take 0.93 - 0.94 of the time.
static bool stays(int64_t bytes) { return bytes <= (int64_t)256 << 20; }
#define PM_STREAM_SWITCH(streams, MODE, STREAM, ...)                                                 \
    do {                                                                                             \
        if (MODE == ROWS_16 && (streams)) { constexpr bool STREAM = MODE == ROWS_16; __VA_ARGS__; }  \
        else { constexpr bool STREAM = false; __VA_ARGS__; }                                         \
    } while (0)

SlotFill slot_fill(void *workspace, const int32_t *indices, const int32_t *locations, int64_t stride, int top_k, int samples, int experts,
                   int capacity, int64_t row_bytes, hipStream_t st)
{
    const int slots = experts * capacity;
    const int64_t pairs = (int64_t)samples * top_k;
    // as many work-groups as have 16 slots each, fewer where each has more to walk (8 bytes a pair, from the caches)
    int shift = 0;
    while (shift < (pairs <= 8192 ? 8 : pairs <= 32768 ? 7 : 6) && (slots >> (shift + 1)) >= 16) ++shift;
    // The walk is as long as the pairs are many, and the rows that hide it are as long as they are wide: the line is fitted between these.
    // Forward pass of the routing API, flags and walk, us: 8000 pairs of 512 bytes 46.8 and 45.1, 6000 of 2048 35.6 and 31.9; 13200 of 512 50.9 and 52.9, 32768 of 1024 41.6 and 47.9, 32768 of 2048 54.5 and 58.4, 20000 of
    // 4096 66.8 and 68.8, 32768 of 4096 99.6 and 100.0; the dispatch alone, rows of 2048 bytes, 12300 pairs 12.6 and 12.5, 16384 14.0 and 13.5, 20480 15.9 and
    // 17.8, 32768 22.8 and 25.3.  A combine's backward pass, whose rows hide more, gains from the walk beyond the line (2048 bytes, 16384 pairs 21.1 and 17.6, 32768
    // 40.8 and 35.6); the line serves both.  With the backward pass 13200 of 4096 130.3 and 125.1, 16384 of 8192 193.8 and 186.4.
    if (pairs <= std::min<int64_t>(8192 + 2 * row_bytes, SLOT_FILL_PAIRS) && (slots >> shift) < SLOT_FILL_BITS) return SlotFill{nullptr, 1 << shift, shift};
    uint32_t *flags = (uint32_t *)workspace;
    slot_flags_clear<<<(slots + 255) / 256, 256, 0, st>>>(flags, slots);
    if (samples > 0)
        slot_flags_mark<<<(samples * top_k + 255) / 256, 256, 0, st>>>(flags, indices, locations, stride,
                                                                      top_k, samples, experts, capacity);
    return SlotFill{flags, std::min((slots + 3) / 4, 2048), 0};
}

int check_planes(const char *who, const int32_t *indices, const int32_t *locations,
                        int64_t stride, int top_k, int samples)
{
    PM_REQUIRE(indices && locations, "%s: indices/locations must not be NULL", who);
    PM_REQUIRE(top_k >= 1, "%s: top_k must be >= 1 (got %d)", who, top_k);
    PM_REQUIRE(samples >= 0, "%s: samples must be >= 0", who);
    PM_REQUIRE(stride >= samples, "%s: plane_stride %lld < samples %d", who, (long long)stride, samples);
    return 0;
}

} // namespace pm

using namespace pm;

extern "C" size_t planmoe_dispatch_workspace_bytes(int experts, int capacity)
{
    if (experts <= 0 || capacity <= 0) return 16;
    return round_up((size_t)experts * (size_t)capacity * sizeof(uint32_t), 256);
}

extern "C" int planmoe_dispatch_fwd(const void *x, int dtype, const float *gates,
                                    const int32_t *indices, const int32_t *locations,
                                    int64_t plane_stride, int top_k, int samples, int model_dim,
                                    int experts, int capacity, void *dispatched, void *workspace,
                                    size_t workspace_bytes, void *stream)
{
    if (check_planes("planmoe_dispatch_fwd", indices, locations, plane_stride, top_k, samples)) return 1;
    PM_REQUIRE(dtype_ok(dtype), "planmoe_dispatch_fwd: bad dtype %d", dtype);
    PM_REQUIRE(model_dim >= 1 && experts >= 1 && capacity >= 0, "planmoe_dispatch_fwd: bad shape");
    PM_REQUIRE((int64_t)experts * capacity < (1ll << 31), "planmoe_dispatch_fwd: experts*capacity overflows int32");
    PM_REQUIRE((int64_t)samples * top_k < (1ll << 31), "planmoe_dispatch_fwd: samples*top_k overflows int32");
    const int slots = experts * capacity;
    if (slots == 0) return 0;
    PM_REQUIRE(x || samples == 0, "planmoe_dispatch_fwd: x is NULL");
    PM_REQUIRE(dispatched, "planmoe_dispatch_fwd: dispatched is NULL");
    PM_REQUIRE(workspace && workspace_bytes >= planmoe_dispatch_workspace_bytes(experts, capacity),
               "planmoe_dispatch_fwd: workspace too small (%zu < %zu)", workspace_bytes,
               planmoe_dispatch_workspace_bytes(experts, capacity));
    hipStream_t st = (hipStream_t)stream;
    const SlotFill fill = slot_fill(workspace, indices, locations, plane_stride, top_k, samples, experts, capacity,
                                    (int64_t)model_dim * (dtype == PLANMOE_F32 ? 4 : 2), st);
    const int token_blocks = (samples + 3) / 4;
    const int mode = rows_mode(dtype, model_dim, x, dispatched);
    const int64_t buffer_bytes = (int64_t)slots * model_dim * (dtype == PLANMOE_F32 ? 4 : 2);
    PM_DTYPE_SWITCH(dtype, DT, {
        PM_ROWS_SWITCH(mode, MODE, PM_STREAM_SWITCH(!stays(buffer_bytes), MODE, STREAM, (dispatch_kernel<DT, MODE, STREAM><<<token_blocks + fill.blocks, 256, 0, st>>>(
            x, gates, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, dispatched, fill,
            token_blocks))));
    });
    PM_LAUNCH_CHECK("planmoe_dispatch_fwd");
    return 0;
}

extern "C" int planmoe_combine_fwd(const void *dispatched, int dtype, const float *gates,
                                   const int32_t *indices, const int32_t *locations,
                                   int64_t plane_stride, int top_k, int samples, int model_dim,
                                   int capacity, void *out, void *stream)
{
    if (check_planes("planmoe_combine_fwd", indices, locations, plane_stride, top_k, samples)) return 1;
    PM_REQUIRE(dtype_ok(dtype), "planmoe_combine_fwd: bad dtype %d", dtype);
    PM_REQUIRE(model_dim >= 1 && capacity >= 0, "planmoe_combine_fwd: bad shape");
    if (samples == 0) return 0;
    PM_REQUIRE(out, "planmoe_combine_fwd: out is NULL");
    PM_REQUIRE(dispatched || capacity == 0, "planmoe_combine_fwd: dispatched is NULL");
    hipStream_t st = (hipStream_t)stream;
    const int mode = rows_mode(dtype, model_dim, out, dispatched);
    const int blocks = (samples + 3) / 4;
    // Eight units a lane: rows above 4 KB, in 16 bits, whose units take twice the registers unpacked, only where the caches do not hold what is moved (14020 x
    // 3528 beside the kernel), or where eight lanes at most have a unit of a row's last pass of four a lane.  us, two choices, bf16 rows that the caches hold, with
    // four and with eight:  1400 tokens x 3876 6.8, 7.5   4000 x 4096 15.9, 17.8   4000 x 2176 10.9, 11.8   8000 x 2304 19.2, 20.9   1400 x 2112 7.0, 5.8
    // fp32:  1400 x 1056 5.5, 4.6   1400 x 2048 5.9, 5.5   4000 x 2560 19.3, 19.5   6800 x 4096 66, 62
    // An element at a time (rows that start anywhere), in bf16:  300 x 3877 10.0, 7.9   2000 x 2051 8.9, 7.9   2000 x 3877 14.7, 11.8   8000 x 2051 19.2, 19.7   14000 x 3877 69, 65
    const int64_t row_bytes = (int64_t)model_dim * (dtype == PLANMOE_F32 ? 4 : 2);
    const bool few_lanes = ((row_bytes + 15) / 16 + 255) % 256 < 8;
    const bool wide = row_bytes > 4096 && (dtype == PLANMOE_F32 || mode == ROWS_1 || few_lanes || !stays(row_bytes * samples * (top_k + 1)));
    // One unit a lane where a wave covers a row with them: more are loads that are thrown away.  us, two choices, four units of one choice at a time, four of two, one of two:
    // 2156 x 64 bf16 4.9, 5.4, 2.8   1514 x 32 fp16 4.7, 6.1, 2.7   12971 x 100 fp32 7.2, 6.5, 4.4   16000 x 512 bf16 11.8, 12.0, 8.4
    const bool narrow = model_dim <= WAVE * (mode == ROWS_1 ? 1 : dtype == PLANMOE_F32 ? 4 : 8);
    if (capacity == 0) {
        // no slot exists, every choice is dropped: zero rows.  (combine_kernel fetches rows with
        // unconditional loads at clamped slots and must not run without a row to read.)
        PM_DTYPE_SWITCH(dtype, DT, {
            PM_ROWS_SWITCH(mode, MODE, (zero_rows_kernel<DT, MODE><<<blocks, 256, 0, st>>>(out, samples, model_dim)));
        });
        PM_LAUNCH_CHECK("planmoe_combine_fwd");
        return 0;
    }
    PM_DTYPE_SWITCH(dtype, DT, {
        PM_ROWS_SWITCH(mode, MODE, ({
            if (narrow) combine_kernel<DT, MODE, 1><<<blocks, 256, 0, st>>>(dispatched, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out);
            else if (wide) combine_kernel<DT, MODE, 8><<<blocks, 256, 0, st>>>(dispatched, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out);
            else combine_kernel<DT, MODE, 4><<<blocks, 256, 0, st>>>(dispatched, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out);
        }));
    });
    PM_LAUNCH_CHECK("planmoe_combine_fwd");
    return 0;
}

extern "C" int planmoe_bwd_gate(const void *x, const void *dispatched, int dtype,
                                const int32_t *indices, const int32_t *locations,
                                int64_t plane_stride, int top_k, int samples, int model_dim,
                                int capacity, float *grad_gates, void *stream)
{
    if (check_planes("planmoe_bwd_gate", indices, locations, plane_stride, top_k, samples)) return 1;
    PM_REQUIRE(dtype_ok(dtype), "planmoe_bwd_gate: bad dtype %d", dtype);
    PM_REQUIRE(model_dim >= 1 && capacity >= 0, "planmoe_bwd_gate: bad shape");
    if (samples == 0) return 0;
    PM_REQUIRE(x && grad_gates, "planmoe_bwd_gate: NULL argument");
    PM_REQUIRE(dispatched || capacity == 0, "planmoe_bwd_gate: dispatched is NULL");
    hipStream_t st = (hipStream_t)stream;
    if (capacity == 0) {                               // no slot, no row to read: every gradient is zero
        for (int j = 0; j < top_k; ++j) fill_u32((uint32_t *)(grad_gates + (int64_t)j * plane_stride), (size_t)samples, 0u, st);
        PM_LAUNCH_CHECK("planmoe_bwd_gate");
        return 0;
    }
    const int mode = rows_mode(dtype, model_dim, x, dispatched);
    const int blocks = (samples + 3) / 4;
    PM_DTYPE_SWITCH(dtype, DT, {
        if (mode == ROWS_16)
            bwd_gate_kernel<DT, ROWS_16><<<blocks, 256, 0, st>>>(
                x, dispatched, indices, locations, plane_stride, top_k, samples, model_dim, capacity, grad_gates);
        else
            bwd_gate_kernel<DT, ROWS_1><<<blocks, 256, 0, st>>>(
                x, dispatched, indices, locations, plane_stride, top_k, samples, model_dim, capacity, grad_gates);
    });
    PM_LAUNCH_CHECK("planmoe_bwd_gate");
    return 0;
}

extern "C" int planmoe_combine_bwd(const void *grad, const void *dispatched, int dtype, const float *gates,
                                   const int32_t *indices, const int32_t *locations, int64_t plane_stride,
                                   int top_k, int samples, int model_dim, int experts, int capacity,
                                   void *grad_dispatched, float *grad_gates, void *workspace,
                                   size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_combine_bwd";
    if (check_planes(who, indices, locations, plane_stride, top_k, samples)) return 1;
    PM_REQUIRE(dtype_ok(dtype), "%s: bad dtype %d", who, dtype);
    PM_REQUIRE(model_dim >= 1 && experts >= 1 && capacity >= 1 && samples >= 1, "%s: bad shape", who);
    PM_REQUIRE((int64_t)experts * capacity < (1ll << 31), "%s: experts*capacity overflows int32", who);
    PM_REQUIRE((int64_t)samples * top_k < (1ll << 31), "%s: samples*top_k overflows int32", who);
    PM_REQUIRE(grad && dispatched && grad_dispatched && grad_gates, "%s: NULL argument", who);
    PM_REQUIRE(workspace && workspace_bytes >= planmoe_dispatch_workspace_bytes(experts, capacity), "%s: workspace too small", who);
    hipStream_t st = (hipStream_t)stream;
    const SlotFill fill = slot_fill(workspace, indices, locations, plane_stride, top_k, samples, experts, capacity,
                                    (int64_t)model_dim * (dtype == PLANMOE_F32 ? 4 : 2), st);
    const int token_blocks = (samples + 3) / 4;
    const int mode = std::min(rows_mode(dtype, model_dim, grad, dispatched), rows_mode(dtype, model_dim, grad_dispatched, grad_dispatched));
    const int64_t buffer_bytes = (int64_t)experts * capacity * model_dim * (dtype == PLANMOE_F32 ? 4 : 2);
    PM_DTYPE_SWITCH(dtype, DT, {
        PM_ROWS_SWITCH(mode, MODE, PM_STREAM_SWITCH(!stays(2 * buffer_bytes), MODE, STREAM, (combine_bwd_kernel<DT, MODE, STREAM><<<token_blocks + fill.blocks, 256, 0, st>>>(
            grad, dispatched, gates, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity,
            grad_dispatched, grad_gates, fill, token_blocks))));
    });
    PM_LAUNCH_CHECK(who);
    return 0;
}
