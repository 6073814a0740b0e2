// The row passes of the layer whose experts' buffers never leave the GPU: combine and its backward
// pass with the codec of the exchange in between.
//
// On one rank the all-to-all delivers what was sent, so what "int8" does to a row is
// decompress(compress(row)) (int8.cpp:10-24, 46-60).  The kernels here apply that to a row while it is
// in registers -- the same roundings, the same values -- instead of writing codes that the next launch
// decodes: the combine reads the experts' rows once (T k M values) where compress, then combine from the
// codes, read E C M values, wrote and read their codes.  Only rows that hold a token are touched: empty
// capacity slots are never written and never read.
#include "rows.hpp"
#include "int8_core.hpp"
#include "layer_rows.hpp"
#include "layer_shares.hpp"
#include "route_bwd.hpp"

#include <type_traits>

namespace pm {

// out[t] = sum_j gate_j * codec(rows[slot_j]), planes left to right, one rounding at the end.
// One wave per token; the rows of two choices are requested before either is used and stay as they lie in
// memory until their values are looked up, vector by vector (two 8 KB rows and their sum in fp32 took 230
// registers and left two waves per SIMD).  16384 x 4096 bf16, top-2, 403 MB: 81 us = 5.0 TB/s.  More than two
// choices keep their sum in fp32.  KEEP: the rows' codes, minima and scales are stored as well, by slot (what a backward
// pass reads in place of the rows: a byte a value to hold between the passes; 16384 x 1024 bf16, top-2: 26.5 -> 32 us, and the
// backward pass 48 -> 38).  SHARES: bf16 rows that the product left in shares; `rows` is not read.
template <int DT, int CACHE, bool TWO, bool KEEP, bool SHARES = false>
__global__ __launch_bounds__(256) void layer_combine_kernel(
    const void *__restrict__ rows, const float *__restrict__ gates, const int32_t *__restrict__ indices,
    const int32_t *__restrict__ locations, int64_t stride, int top_k, int samples, int model_dim, int capacity,
    void *__restrict__ out, uint8_t *__restrict__ codes, void *__restrict__ bias, void *__restrict__ scales, const RowShares shares = RowShares{})
{
    using E = Elem<DT>;
    constexpr int V = E::VEC;
    __shared__ __align__(16) float s_table[4][2][256];
    const int lane = lane_id(), units = model_dim / V;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= samples) return;                    // (no work-group barrier below)
    const int64_t row_bytes = (int64_t)model_dim * (int64_t)sizeof(typename E::store_t);
    uint4 *dst = reinterpret_cast<uint4 *>((char *)out + (int64_t)t * row_bytes);
    auto request = [&](int s, uint4 (&r)[CACHE]) {
        if constexpr (SHARES) {
#pragma unroll
            for (int c = 0; c < CACHE; ++c) r[c] = shares.vector(max(s, 0), min(c * WAVE + lane, units - 1));
            return;
        }
        const uint4 *src = reinterpret_cast<const uint4 *>((const char *)rows + (int64_t)max(s, 0) * row_bytes);
#pragma unroll
        for (int c = 0; c < CACHE; ++c) r[c] = src[min(c * WAVE + lane, units - 1)];
    };
    auto keep_codes = [&](int s, int c, const CodeWords<DT> &code) {
        if (KEEP && s >= 0 && c * WAVE + lane < units) store_codes<DT>(codes + (int64_t)s * model_dim + (c * WAVE + lane) * V, code);
    };
    auto keep_row = [&](int s, float mn, float scale) {
        if (KEEP && s >= 0 && lane == 0) { E::store(bias, s, mn); E::store(scales, s, scale); }
    };
    if constexpr (TWO) {
        int slot; float gate;
        fetch_planes(gates, indices, locations, stride, t, 0, top_k, 0x7fffffff, capacity, slot, gate);
        uint4 r0[CACHE], r1[CACHE];
        const int s0 = rl_i(slot, 0), s1 = top_k > 1 ? rl_i(slot, 1) : -1;
        const float g0 = rl_f(gate, 0), g1 = rl_f(gate, 1);
        request(s0, r0);
        if (s1 >= 0) request(s1, r1);
        const RowTable<DT> t0(r0, g0, s_table[threadIdx.x >> 6][0]);
        // (a choice without a slot has no row: row 0 stands for it above, what is looked up is not used)
        const RowTable<DT> t1(s1 >= 0 ? r1 : r0, g1, s_table[threadIdx.x >> 6][1]);
        table_sync();
        keep_row(s0, t0.mn, t0.scale);
        keep_row(s1, t1.mn, t1.scale);
        auto body = [&](auto mode) {
#pragma unroll
            for (int c = 0; c < CACHE; ++c) {
                float f[V], h[V];
                t0.template values<decltype(mode)::value>(r0[c], f, [&](const CodeWords<DT> &code) { keep_codes(s0, c, code); });
#pragma unroll
                for (int i = 0; i < V; ++i) f[i] = s0 >= 0 ? f[i] : 0.f;
                if (top_k > 1) {
                    if (s1 >= 0) {
                        t1.template values<decltype(mode)::value>(r1[c], h, [&](const CodeWords<DT> &code) { keep_codes(s1, c, code); });
#pragma unroll
                        for (int i = 0; i < V; ++i) f[i] += h[i];
                    } else {
#pragma unroll
                        for (int i = 0; i < V; ++i) f[i] += 0.f;
                    }
                }
                if (c * WAVE + lane < units) stream_store(dst + c * WAVE + lane, E::pack(f));
            }
        };
        if (t0.enc.fast() && t1.enc.fast()) body(std::true_type{}); else body(std::false_type{});
        return;
    }
    float acc[CACHE][V];
    for (int j0 = 0; j0 < top_k; j0 += WAVE) {
        const int np = min(top_k - j0, WAVE);
        int slot; float gate;
        fetch_planes(gates, indices, locations, stride, t, j0, np, 0x7fffffff, capacity, slot, gate);
        for (int j = 0; j < np; ++j) {
            uint4 r[CACHE];
            const int s = rl_i(slot, j);
            const float g = rl_f(gate, j);
            request(s, r);
            if (s >= 0) {
                const float2 row = through_int8<DT, CACHE, false>(r, [&](int c, const CodeWords<DT> &code) { keep_codes(s, c, code); });
                keep_row(s, row.x, row.y);
            }
#pragma unroll
            for (int c = 0; c < CACHE; ++c) {
                float f[V];
                E::unpack(r[c], f);
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const float v = s >= 0 ? g * f[i] : 0.f;
                    acc[c][i] = j0 + j == 0 ? v : acc[c][i] + v;
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < CACHE; ++c) if (c * WAVE + lane < units) stream_store(dst + c * WAVE + lane, E::pack(acc[c]));
}

// Backward of the combine: grad_gates_j = <grad[t], codec(rows[slot_j])> and grad_rows[slot_j] =
// codec(round(gate_j * grad[t])) (GatingDecoder.backward, fast_dispatch.py:62-79, with the two codec
// passes around it, overlap.py:19-34).  The rows come as they are (SEEN_ROWS without a codec, SEEN_INT8 with), or as the codes,
// minima and scales that the forward pass kept (SEEN_CODES): half or a quarter of the bytes, and no codes to work out.
// 16384 x 1024 bf16, top-2: 48 us from the rows, 38 from the codes (33 MB of the gradient in, 34 of codes, 67 out).
// grad_logits given: up to 64 choices, whose gates' gradients go on through the routing into the logits' while the wave has them, and
// grad_gates is not written (a launch of its own reads and writes 100 bytes a token: 5 us, and as much of the host's time).
enum { SEEN_ROWS, SEEN_INT8, SEEN_CODES };
template <int DT, int CACHE, int SEEN>
__global__ __launch_bounds__(256) void layer_combine_bwd_kernel(
    const void *__restrict__ grad, const void *__restrict__ rows, const void *__restrict__ bias, const void *__restrict__ scales,
    const float *__restrict__ gates, const int32_t *__restrict__ indices, const int32_t *__restrict__ locations, int64_t stride,
    int top_k, int samples, int model_dim, int capacity, void *__restrict__ grad_rows, float *__restrict__ grad_gates,
    const RouteBwd route, int scores_dtype, float *__restrict__ grad_logits)
{
    using E = Elem<DT>;
    constexpr int V = E::VEC;
    __shared__ __align__(16) float s_table[4][256];
    const int lane = lane_id(), units = model_dim / V;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= samples) return;                    // (no work-group barrier below)
    const int64_t row_bytes = (int64_t)model_dim * (int64_t)sizeof(typename E::store_t);
    constexpr bool INT8 = SEEN != SEEN_ROWS;
    using seen_t = std::conditional_t<SEEN == SEEN_CODES, CodeWords<DT>, uint4>;       // a lane's vector of a row
    uint4 g_row[CACHE];
    {
        const uint4 *src = reinterpret_cast<const uint4 *>((const char *)grad + (int64_t)t * row_bytes);
#pragma unroll
        for (int c = 0; c < CACHE; ++c) g_row[c] = src[min(c * WAVE + lane, units - 1)];
    }
    float dgate = 0.f;                           // lane j: the gradient of gate j
    for (int j0 = 0; j0 < top_k; j0 += WAVE) {
        const int np = min(top_k - j0, WAVE);
        int slot; float gate;
        fetch_planes(gates, indices, locations, stride, t, j0, np, 0x7fffffff, capacity, slot, gate);
        if (grad_gates && lane < np && slot < 0) grad_gates[(int64_t)(j0 + lane) * stride + t] = 0.f;
        float mn = 0.f, scale = 0.f;
        if (SEEN == SEEN_CODES && lane < np && slot >= 0) { mn = E::load(bias, slot); scale = E::load(scales, slot); }
        // the next choice's row is on its way while this one's is worked on (a dropped choice reads slot 0, unused)
        seen_t next[CACHE];
        auto request = [&](int j) {
            const seen_t *src = reinterpret_cast<const seen_t *>(rows) + (int64_t)max(rl_i(slot, j), 0) * units;
#pragma unroll
            for (int c = 0; c < CACHE; ++c) next[c] = src[min(c * WAVE + lane, units - 1)];
        };
        request(0);
        for (int j = 0; j < np; ++j) {
            const int s = rl_i(slot, j);
            const float g = rl_f(gate, j);
            seen_t seen[CACHE];
#pragma unroll
            for (int c = 0; c < CACHE; ++c) seen[c] = next[c];
            if (j + 1 < np) request(j + 1);
            if (s < 0) continue;
            float acc = 0.f;
            auto dot = [&](int c, const float (&b)[V]) {
                float a[V];
                E::unpack(g_row[c], a);
                if (c * WAVE + lane < units) {
#pragma unroll
                    for (int i = 0; i < V; ++i) acc = fmaf(b[i], a[i], acc);
                }
            };
            if constexpr (SEEN == SEEN_CODES) {
                float *table = s_table[threadIdx.x >> 6];
                fill_table<DT>(rl_f(mn, j), rl_f(scale, j), 1.f, table);
                table_sync();
#pragma unroll
                for (int c = 0; c < CACHE; ++c) {
                    float b[V];
#pragma unroll
                    for (int i = 0; i < V; ++i) b[i] = table[(seen[c].w[i / 4] >> (8 * (i % 4))) & 0xffu];
                    dot(c, b);
                }
                table_sync();
            } else if constexpr (SEEN == SEEN_INT8) {
                float *table = s_table[threadIdx.x >> 6];
                const RowTable<DT> tab(seen, 1.f, table);
                table_sync();
                auto body = [&](auto mode) {
#pragma unroll
                    for (int c = 0; c < CACHE; ++c) {
                        float b[V];
                        tab.template values<decltype(mode)::value>(seen[c], b);
                        dot(c, b);
                    }
                };
                if (tab.enc.fast()) body(std::true_type{}); else body(std::false_type{});
                table_sync();
            } else {
#pragma unroll
                for (int c = 0; c < CACHE; ++c) {
                    float b[V];
                    E::unpack(seen[c], b);
                    dot(c, b);
                }
            }
            acc = wave_sum(acc);
            if (grad_gates && lane == 0) grad_gates[(int64_t)(j0 + j) * stride + t] = acc;
            if (lane == j) dgate = acc;
            // the gradient row as the dispatcher stores it for this gate: round(0 + g * x)
            uint4 r[CACHE];
#pragma unroll
            for (int c = 0; c < CACHE; ++c) {
                float a[V];
                E::unpack(g_row[c], a);
#pragma unroll
                for (int i = 0; i < V; ++i) a[i] = E::round(0.f + g * a[i]);
                r[c] = E::pack(a);
            }
            uint4 *dst = reinterpret_cast<uint4 *>((char *)grad_rows + (int64_t)s * row_bytes);
            if constexpr (INT8) {
                const RowTable<DT> tab(r, 1.f, s_table[threadIdx.x >> 6]);
                table_sync();
                auto body = [&](auto mode) {
#pragma unroll
                    for (int c = 0; c < CACHE; ++c) {
                        float b[V];
                        tab.template values<decltype(mode)::value>(r[c], b);
                        if (c * WAVE + lane < units) stream_store(dst + c * WAVE + lane, E::pack(b));
                    }
                };
                if (tab.enc.fast()) body(std::true_type{}); else body(std::false_type{});
                table_sync();                    // (the next choice's table takes this one's place)
            } else {
#pragma unroll
                for (int c = 0; c < CACHE; ++c) if (c * WAVE + lane < units) stream_store(dst + c * WAVE + lane, r[c]);
            }
        }
    }
    if (grad_logits) {
        const int at = lane < top_k ? indices[(int64_t)lane * stride + t] : -1;
        auto logits = [&](auto dt) {
            constexpr int ST = decltype(dt)::value;
            route_bwd_token<ST>(route, t, lane % route.group, true, [&](int j) { return rl_i(at, j); },
                                [&](int j) { return Elem<ST>::round(rl_f(dgate, j)); },
                                [&](int e, float v) { if (lane < route.group) grad_logits[(int64_t)t * route.experts + e] = Elem<ST>::round(v); });
        };
        if (scores_dtype == PLANMOE_F32) logits(std::integral_constant<int, PLANMOE_F32>{});
        else if (scores_dtype == PLANMOE_BF16) logits(std::integral_constant<int, PLANMOE_BF16>{});
        else logits(std::integral_constant<int, PLANMOE_F16>{});
    }
}

} // namespace pm

using namespace pm;

namespace pm {

int layer_rows_check(const char *who, int dtype, const void *rows, const int32_t *indices, const int32_t *locations, int64_t stride,
                     int top_k, int samples, int model_dim, int experts, int capacity, int codec)
{
    if (check_planes(who, indices, locations, stride, top_k, samples)) return 1;
    PM_REQUIRE(dtype_ok(dtype), "%s: bad dtype %d", who, dtype);
    PM_REQUIRE(codec == 0 || codec == 1, "%s: codec is 0 (none) or 1 (int8)", who);
    const int vec = dtype == PLANMOE_F32 ? 4 : 8;
    PM_REQUIRE(model_dim >= 1 && model_dim % vec == 0 && model_dim <= 16 * WAVE * vec,
               "%s: model_dim must be a multiple of %d, at most %d", who, vec, 16 * WAVE * vec);
    PM_REQUIRE(capacity >= 1 && experts >= 1 && (int64_t)experts * capacity < (1ll << 31), "%s: bad capacity", who);
    PM_REQUIRE((rows && aligned16(rows)) || samples == 0, "%s: NULL or unaligned rows", who);
    return 0;
}

} // namespace pm

// codes NULL: none are kept
static int combine_int8_rows(const char *who, const void *rows, int dtype, const float *gates, const int32_t *indices, const int32_t *locations,
                             int64_t plane_stride, int top_k, int samples, int model_dim, int capacity, void *out, uint8_t *codes, void *bias,
                             void *scale, void *stream)
{
    if (samples == 0) return 0;
    PM_REQUIRE(out && aligned16(out), "%s: NULL or unaligned output", who);
    const int per_lane = (model_dim / (dtype == PLANMOE_F32 ? 4 : 8) + WAVE - 1) / WAVE;
    hipStream_t st = (hipStream_t)stream;
#define PM_LC_(CACHE, TWO, KEEP) (layer_combine_kernel<DT, CACHE, TWO, KEEP><<<(samples + 3) / 4, 256, 0, st>>>(rows, gates, indices, locations, \
        plane_stride, top_k, samples, model_dim, capacity, out, codes, bias, scale))
#define PM_LC(CACHE)                                                                          \
    do {                                                                                      \
        if (top_k <= 2) { if (codes) PM_LC_(CACHE, true, true); else PM_LC_(CACHE, true, false); }     \
        else { if (codes) PM_LC_(CACHE, false, true); else PM_LC_(CACHE, false, false); }     \
    } while (0)
    PM_DTYPE_SWITCH(dtype, DT, PM_ROW_CACHE(PM_LC));
#undef PM_LC
#undef PM_LC_
    PM_LAUNCH_CHECK(who);
    return 0;
}

int pm::combine_int8_shares(const char *who, const RowShares &rows, const float *gates, const int32_t *indices, const int32_t *locations, int64_t plane_stride,
                            int top_k, int samples, void *out, uint8_t *codes, void *bias, void *scale, hipStream_t st)
{
    const int per_lane = (rows.model_dim / 8 + WAVE - 1) / WAVE;
#define PM_LS_(CACHE, TWO, KEEP) (layer_combine_kernel<PLANMOE_BF16, CACHE, TWO, KEEP, true><<<(samples + 3) / 4, 256, 0, st>>>(nullptr, gates, indices, locations, \
        plane_stride, top_k, samples, rows.model_dim, rows.capacity, out, codes, bias, scale, rows))
#define PM_LS(CACHE)                                                                          \
    do {                                                                                      \
        if (top_k <= 2) { if (codes) PM_LS_(CACHE, true, true); else PM_LS_(CACHE, true, false); }     \
        else { if (codes) PM_LS_(CACHE, false, true); else PM_LS_(CACHE, false, false); }     \
    } while (0)
    if (per_lane <= 1) PM_LS(1);
    else if (per_lane <= 2) PM_LS(2);
    else if (per_lane <= 4) PM_LS(4);
    else PM_LS(8);
#undef PM_LS
#undef PM_LS_
    PM_LAUNCH_CHECK(who);
    return 0;
}

extern "C" int planmoe_layer_combine(const void *rows, int dtype, int codec, const float *gates, const int32_t *indices,
                                     const int32_t *locations, int64_t plane_stride, int top_k, int samples, int model_dim,
                                     int experts, int capacity, void *out, void *stream)
{
    const char *who = "planmoe_layer_combine";
    if (layer_rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, codec)) return 1;
    if (codec == 0) return planmoe_combine_fwd(rows, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out, stream);
    return combine_int8_rows(who, rows, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out, nullptr, nullptr,
                             nullptr, stream);
}

extern "C" int planmoe_layer_combine_keep(const void *rows, int dtype, const float *gates, const int32_t *indices, const int32_t *locations,
                                          int64_t plane_stride, int top_k, int samples, int model_dim, int experts, int capacity,
                                          void *out, uint8_t *codes, void *bias, void *scale, void *stream)
{
    const char *who = "planmoe_layer_combine_keep";
    if (layer_rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, 1)) return 1;
    PM_REQUIRE(codes && bias && scale && aligned16(codes), "%s: NULL output, or codes not 16-byte aligned", who);
    return combine_int8_rows(who, rows, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out, codes, bias, scale,
                             stream);
}

// seen: SEEN_ROWS, SEEN_INT8 or SEEN_CODES (bias and scale are read with the last only)
static int combine_bwd_rows(const char *who, int seen, const void *grad, const void *rows, const void *bias, const void *scale, int dtype,
                            const float *gates, const int32_t *indices, const int32_t *locations, int64_t plane_stride, int top_k,
                            int samples, int model_dim, int capacity, void *grad_rows, float *grad_gates, void *stream,
                            const RouteBwd &route = RouteBwd{}, int scores_dtype = 0, float *grad_logits = nullptr)
{
    if (samples == 0) return 0;
    PM_REQUIRE(grad && grad_rows && (grad_gates || grad_logits) && gates && aligned16(grad) && aligned16(grad_rows), "%s: NULL or unaligned argument", who);
    const int per_lane = (model_dim / (dtype == PLANMOE_F32 ? 4 : 8) + WAVE - 1) / WAVE;
    hipStream_t st = (hipStream_t)stream;
#define PM_LB_(CACHE, SEEN) (layer_combine_bwd_kernel<DT, CACHE, SEEN><<<(samples + 3) / 4, 256, 0, st>>>(grad, rows, bias, scale, gates, indices, \
        locations, plane_stride, top_k, samples, model_dim, capacity, grad_rows, grad_gates, route, scores_dtype, grad_logits))
#define PM_LB(CACHE)                                                                          \
    do {                                                                                      \
        if (seen == SEEN_CODES) PM_LB_(CACHE, SEEN_CODES);                                    \
        else if (seen == SEEN_INT8) PM_LB_(CACHE, SEEN_INT8);                                 \
        else PM_LB_(CACHE, SEEN_ROWS);                                                        \
    } while (0)
    PM_DTYPE_SWITCH(dtype, DT, PM_ROW_CACHE(PM_LB));
#undef PM_LB
#undef PM_LB_
    PM_LAUNCH_CHECK(who);
    return 0;
}

extern "C" int planmoe_layer_combine_bwd(const void *grad, const void *rows, int dtype, int codec, const float *gates,
                                         const int32_t *indices, const int32_t *locations, int64_t plane_stride, int top_k,
                                         int samples, int model_dim, int experts, int capacity, void *grad_rows,
                                         float *grad_gates, void *stream)
{
    const char *who = "planmoe_layer_combine_bwd";
    if (layer_rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, codec)) return 1;
    return combine_bwd_rows(who, codec ? SEEN_INT8 : SEEN_ROWS, grad, rows, nullptr, nullptr, dtype, gates, indices, locations, plane_stride, top_k,
                            samples, model_dim, capacity, grad_rows, grad_gates, stream);
}

extern "C" int planmoe_layer_combine_bwd_codes(const void *grad, const uint8_t *codes, const void *bias, const void *scale, int dtype,
                                               const float *gates, const int32_t *indices, const int32_t *locations,
                                               int64_t plane_stride, int top_k, int samples, int model_dim, int experts,
                                               int capacity, void *grad_rows, float *grad_gates, void *stream)
{
    const char *who = "planmoe_layer_combine_bwd_codes";
    if (layer_rows_check(who, dtype, codes, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, 1)) return 1;
    PM_REQUIRE((bias && scale) || samples == 0, "%s: NULL argument", who);
    return combine_bwd_rows(who, SEEN_CODES, grad, codes, bias, scale, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim,
                            capacity, grad_rows, grad_gates, stream);
}

extern "C" int planmoe_layer_combine_bwd_logits(const void *grad, const void *rows, const void *bias, const void *scale, int dtype, int codec,
                                                const float *gates, const int32_t *indices, const int32_t *locations, int64_t plane_stride,
                                                int top_k, int samples, int model_dim, int experts, int capacity, void *grad_rows,
                                                const void *scores, int scores_dtype, int normalize_gate, const float *grad_l_aux,
                                                const int32_t *first_choice_counts, float *grad_logits, void *stream)
{
    const char *who = "planmoe_layer_combine_bwd_logits";
    if (layer_rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, codec)) return 1;
    PM_REQUIRE(dtype_ok(scores_dtype) && top_k <= WAVE && top_k <= experts, "%s: bad scores dtype, or more than %d choices", who, WAVE);
    PM_REQUIRE(codec == 0 || (bias && scale) || samples == 0, "%s: NULL argument", who);
    PM_REQUIRE((scores && grad_logits && (!grad_l_aux || first_choice_counts)) || samples == 0, "%s: NULL argument", who);
    const RouteBwd route{scores, grad_l_aux, grad_l_aux ? first_choice_counts : nullptr, samples, experts, top_k, normalize_gate, route_bwd_group(experts)};
    return combine_bwd_rows(who, codec ? SEEN_CODES : SEEN_ROWS, grad, rows, bias, scale, dtype, gates, indices, locations, plane_stride, top_k, samples,
                            model_dim, capacity, grad_rows, nullptr, stream, route, scores_dtype, grad_logits);
}
