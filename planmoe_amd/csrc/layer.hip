// The row passes of the layer whose experts' buffers never leave the GPU: combine and its backward
// pass with the codec of the exchange in between, and the small reductions of the backward pass.
//
// On one rank the all-to-all delivers what was sent, so what "int8" does to a row is
// decompress(compress(row)) (int8.cpp:10-24, 46-60).  The kernels here apply that to a row while it is
// in registers -- the same roundings, the same values -- instead of writing codes that the next launch
// decodes: the combine reads the experts' rows once (T k M values) where compress, then combine from the
// codes, read E C M values, wrote and read their codes.  Only rows that hold a token are touched: empty
// capacity slots are never written and never read.
#include "rows.hpp"
#include <type_traits>
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

// out[t] = sum_j gate_j * codec(rows[slot_j]), planes left to right, one rounding at the end.
// One wave per token; the rows of two choices are requested before either is used and stay as they lie in
// memory until their values are looked up, vector by vector (two 8 KB rows and their sum in fp32 took 230
// registers and left two waves per SIMD).  16384 x 4096 bf16, top-2, 403 MB: 81 us = 5.0 TB/s.  More than two
// choices keep their sum in fp32.  KEEP: the rows' codes, minima and scales are stored as well, by slot (what a backward
// pass reads in place of the rows: a byte a value to hold between the passes; 16384 x 1024 bf16, top-2: 26.5 -> 32 us, and the
// backward pass 48 -> 38).
template <int DT, int CACHE, bool TWO, bool KEEP>
__global__ __launch_bounds__(256) void layer_combine_kernel(
    const void *__restrict__ rows, const float *__restrict__ gates, const int32_t *__restrict__ indices,
    const int32_t *__restrict__ locations, int64_t stride, int top_k, int samples, int model_dim, int capacity,
    void *__restrict__ out, uint8_t *__restrict__ codes, void *__restrict__ bias, void *__restrict__ scales)
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
enum { SEEN_ROWS, SEEN_INT8, SEEN_CODES };
template <int DT, int CACHE, int SEEN>
__global__ __launch_bounds__(256) void layer_combine_bwd_kernel(
    const void *__restrict__ grad, const void *__restrict__ rows, const void *__restrict__ bias, const void *__restrict__ scales,
    const float *__restrict__ gates, const int32_t *__restrict__ indices, const int32_t *__restrict__ locations, int64_t stride,
    int top_k, int samples, int model_dim, int capacity, void *__restrict__ grad_rows, float *__restrict__ grad_gates)
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
    for (int j0 = 0; j0 < top_k; j0 += WAVE) {
        const int np = min(top_k - j0, WAVE);
        int slot; float gate;
        fetch_planes(gates, indices, locations, stride, t, j0, np, 0x7fffffff, capacity, slot, gate);
        if (lane < np && slot < 0) grad_gates[(int64_t)(j0 + lane) * stride + t] = 0.f;
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
            if (lane == 0) grad_gates[(int64_t)(j0 + j) * stride + t] = acc;
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
}

// Column sums of the rows in use of every batch: out[e][n] = sum_{r < rows_e} a[e][r][n] (the bias gradient).
// A work-group takes 64 vectors of columns and a share of the rows, four rows at a time side by side; the
// shares' sums go to `parts` and the second kernel adds them in order.
template <int DT>
__global__ __launch_bounds__(256) void rows_colsum_kernel(const void *__restrict__ a, const int *__restrict__ live, int live_planes,
                                                          int live_round, int batches, int rows, int cols, int shares, float *__restrict__ parts)
{
    using E = Elem<DT>;
    constexpr int V = E::VEC;
    __shared__ float s_sum[4][WAVE][V + 1];
    const int e = blockIdx.z, share = blockIdx.y, lane = lane_id(), wave = threadIdx.x >> 6;
    const int units = cols / V, u = blockIdx.x * WAVE + lane, uc = min(u, units - 1);
    int used = rows;
    if (live) {
        int n = 0;
        for (int j = 0; j < live_planes; ++j) n += live[j * batches + e];
        used = min(rows, (n + live_round - 1) / live_round * live_round);
    }
    const int per = (used + shares - 1) / shares, r0 = share * per, r1 = min(used, r0 + per);
    const uint4 *src = reinterpret_cast<const uint4 *>((const char *)a + (int64_t)e * rows * cols * (int64_t)sizeof(typename E::store_t));
    float acc[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.f;
    constexpr int R = 4;
    for (int r = r0 + wave * R; r < r1; r += 4 * R) {
        uint4 v[R];
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = src[(int64_t)min(r + q, r1 - 1) * units + uc];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            float f[V];
            E::unpack(v[q], f);
#pragma unroll
            for (int i = 0; i < V; ++i) acc[i] += r + q < r1 ? f[i] : 0.f;
        }
    }
#pragma unroll
    for (int i = 0; i < V; ++i) s_sum[wave][lane][i] = acc[i];
    __syncthreads();
    for (int x = threadIdx.x; x < WAVE * V; x += 256) {
        const int l = x / V, i = x % V, col = (blockIdx.x * WAVE + l) * V + i;
        if (col < cols) parts[((int64_t)e * shares + share) * cols + col] = s_sum[0][l][i] + s_sum[1][l][i] + s_sum[2][l][i] + s_sum[3][l][i];
    }
}

// out[e][c] = sum over the shares, in order within a wave's quarter: 64 columns per work-group, eight loads in flight
// (a thread per column that walked the shares one by one took 35 us for 256 shares of 8 x 1024)
template <int DT>
__global__ __launch_bounds__(256) void parts_sum_kernel(const float *__restrict__ parts, int shares, int cols, void *__restrict__ out)
{
    __shared__ float s_sum[4][WAVE];
    const int e = blockIdx.y, lane = lane_id(), wave = threadIdx.x >> 6, c = blockIdx.x * WAVE + lane;
    const float *from = parts + (int64_t)e * shares * cols + min(c, cols - 1);
    const int per = (shares + 3) / 4, i1 = min(shares, (wave + 1) * per);
    float s = 0.f;
    for (int i = wave * per; i < i1; i += 8) {
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = from[(int64_t)min(i + q, i1 - 1) * cols];
#pragma unroll
        for (int q = 0; q < 8; ++q) s += i + q < i1 ? v[q] : 0.f;
    }
    s_sum[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && c < cols) Elem<DT>::store(out, (int64_t)e * cols + c, s_sum[0][lane] + s_sum[1][lane] + s_sum[2][lane] + s_sum[3][lane]);
}

// Gate weight gradient: parts[share][e][m] = sum_{t in share} g[t][e] * x[t][m]; a work-group takes 64 vectors
// of columns and a share of the tokens, its waves every fourth token; EP experts per pass.
template <int DT, int EP>
__global__ __launch_bounds__(256) void gate_dw_kernel(const void *__restrict__ x, const float *__restrict__ g, int samples, int model_dim,
                                                      int experts, int e0, int shares, float *__restrict__ parts)
{
    using E = Elem<DT>;
    constexpr int V = E::VEC;
    __shared__ float s_sum[3][WAVE][EP * V + 1];
    const int share = blockIdx.y, lane = lane_id(), wave = threadIdx.x >> 6;
    const int units = model_dim / V, u = blockIdx.x * WAVE + lane, uc = min(u, units - 1);
    const int per = (samples + shares - 1) / shares, t0 = share * per, t1 = min(samples, t0 + per);
    const uint4 *src = reinterpret_cast<const uint4 *>(x);
    float acc[EP][V];
#pragma unroll
    for (int e = 0; e < EP; ++e)
#pragma unroll
        for (int i = 0; i < V; ++i) acc[e][i] = 0.f;
    constexpr int R = 4;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    for (int t = t0 + wave_u * R; t < t1; t += 4 * R) {
        uint4 v[R];
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = src[(int64_t)min(t + q, t1 - 1) * units + uc];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            float f[V];
            E::unpack(v[q], f);
            const int tq = min(t + q, t1 - 1);
#pragma unroll
            for (int e = 0; e < EP; ++e) {
                // (uniform: scalar loads; g rounded to x's dtype first, as the cast before a library GEMM would)
                const float ge = e0 + e < experts && t + q < t1 ? E::round(g[(int64_t)tq * experts + e0 + e]) : 0.f;
#pragma unroll
                for (int i = 0; i < V; ++i) acc[e][i] = fmaf(ge, f[i], acc[e][i]);
            }
        }
    }
    if (wave > 0)
#pragma unroll
        for (int e = 0; e < EP; ++e)
#pragma unroll
            for (int i = 0; i < V; ++i) s_sum[wave - 1][lane][e * V + i] = acc[e][i];
    __syncthreads();
    if (wave == 0 && u < units) {
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            if (e0 + e >= experts) break;
            float *to = parts + ((int64_t)share * experts + e0 + e) * model_dim + (int64_t)u * V;
#pragma unroll
            for (int i = 0; i < V; ++i)
                to[i] = acc[e][i] + s_sum[0][lane][e * V + i] + s_sum[1][lane][e * V + i] + s_sum[2][lane][e * V + i];
        }
    }
}

} // namespace pm

using namespace pm;

namespace {

int rows_check(const char *who, int dtype, const void *rows, const int32_t *indices, const int32_t *locations, int64_t stride,
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

}  // namespace

// the rows a wave keeps in registers: 1, 2, 4, 8 or 16 vectors per lane
#define PM_ROW_CACHE(CALL)                                    \
    do {                                                      \
        if (per_lane <= 1) CALL(1);                           \
        else if (per_lane <= 2) CALL(2);                      \
        else if (per_lane <= 4) CALL(4);                      \
        else if (per_lane <= 8) CALL(8);                      \
        else CALL(16);                                        \
    } while (0)

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

extern "C" int planmoe_layer_combine(const void *rows, int dtype, int codec, const float *gates, const int32_t *indices,
                                     const int32_t *locations, int64_t plane_stride, int top_k, int samples, int model_dim,
                                     int experts, int capacity, void *out, void *stream)
{
    const char *who = "planmoe_layer_combine";
    if (rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, codec)) return 1;
    if (codec == 0) return planmoe_combine_fwd(rows, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out, stream);
    return combine_int8_rows(who, rows, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out, nullptr, nullptr,
                             nullptr, stream);
}

extern "C" int planmoe_layer_combine_keep(const void *rows, int dtype, const float *gates, const int32_t *indices, const int32_t *locations,
                                          int64_t plane_stride, int top_k, int samples, int model_dim, int experts, int capacity,
                                          void *out, uint8_t *codes, void *bias, void *scale, void *stream)
{
    const char *who = "planmoe_layer_combine_keep";
    if (rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, 1)) return 1;
    PM_REQUIRE(codes && bias && scale && aligned16(codes), "%s: NULL output, or codes not 16-byte aligned", who);
    return combine_int8_rows(who, rows, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim, capacity, out, codes, bias, scale,
                             stream);
}

// seen: SEEN_ROWS, SEEN_INT8 or SEEN_CODES (bias and scale are read with the last only)
static int combine_bwd_rows(const char *who, int seen, const void *grad, const void *rows, const void *bias, const void *scale, int dtype,
                            const float *gates, const int32_t *indices, const int32_t *locations, int64_t plane_stride, int top_k,
                            int samples, int model_dim, int capacity, void *grad_rows, float *grad_gates, void *stream)
{
    if (samples == 0) return 0;
    PM_REQUIRE(grad && grad_rows && grad_gates && gates && aligned16(grad) && aligned16(grad_rows), "%s: NULL or unaligned argument", who);
    const int per_lane = (model_dim / (dtype == PLANMOE_F32 ? 4 : 8) + WAVE - 1) / WAVE;
    hipStream_t st = (hipStream_t)stream;
#define PM_LB_(CACHE, SEEN) (layer_combine_bwd_kernel<DT, CACHE, SEEN><<<(samples + 3) / 4, 256, 0, st>>>(grad, rows, bias, scale, gates, indices, \
        locations, plane_stride, top_k, samples, model_dim, capacity, grad_rows, grad_gates))
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
    if (rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, codec)) return 1;
    return combine_bwd_rows(who, codec ? SEEN_INT8 : SEEN_ROWS, grad, rows, nullptr, nullptr, dtype, gates, indices, locations, plane_stride, top_k,
                            samples, model_dim, capacity, grad_rows, grad_gates, stream);
}

extern "C" int planmoe_layer_combine_bwd_codes(const void *grad, const uint8_t *codes, const void *bias, const void *scale, int dtype,
                                               const float *gates, const int32_t *indices, const int32_t *locations,
                                               int64_t plane_stride, int top_k, int samples, int model_dim, int experts,
                                               int capacity, void *grad_rows, float *grad_gates, void *stream)
{
    const char *who = "planmoe_layer_combine_bwd_codes";
    if (rows_check(who, dtype, codes, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, 1)) return 1;
    PM_REQUIRE((bias && scale) || samples == 0, "%s: NULL argument", who);
    return combine_bwd_rows(who, SEEN_CODES, grad, codes, bias, scale, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim,
                            capacity, grad_rows, grad_gates, stream);
}

// how many shares a reduction over `rows` is cut into for `blocks` column blocks: enough work-groups for the GPU, at least 32 rows each
static int reduction_shares(int64_t rows, int64_t blocks)
{
    int64_t s = (1024 + blocks - 1) / blocks;
    if (s > (rows + 31) / 32) s = (rows + 31) / 32;
    return (int)(s < 1 ? 1 : s > 256 ? 256 : s);
}

extern "C" size_t planmoe_rows_colsum_workspace_bytes(int batches, int rows, int cols)
{
    if (batches < 1 || rows < 1 || cols < 1) return 16;
    return (size_t)batches * reduction_shares(rows, (int64_t)batches * ((cols + 255) / 256)) * cols * 4;
}

extern "C" int planmoe_rows_colsum(const void *a, int dtype, int batches, int rows, int cols, const int32_t *live, int live_planes,
                                   int live_round, void *out, void *workspace, size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_rows_colsum";
    PM_REQUIRE(dtype_ok(dtype) && batches >= 1 && rows >= 1 && cols >= 1, "%s: bad shape", who);
    const int vec = dtype == PLANMOE_F32 ? 4 : 8;
    PM_REQUIRE(cols % vec == 0 && a && out && aligned16(a), "%s: cols must be a multiple of %d, the rows 16-byte aligned", who, vec);
    PM_REQUIRE(batches < 65536 && (!live || (live_planes >= 1 && live_round >= 1)), "%s: bad live rows", who);
    PM_REQUIRE(workspace && workspace_bytes >= planmoe_rows_colsum_workspace_bytes(batches, rows, cols), "%s: workspace too small", who);
    const int shares = reduction_shares(rows, (int64_t)batches * ((cols + 255) / 256));
    const dim3 grid((unsigned)((cols / vec + WAVE - 1) / WAVE), (unsigned)shares, (unsigned)batches);
    hipStream_t st = (hipStream_t)stream;
    PM_DTYPE_SWITCH(dtype, DT,
        (rows_colsum_kernel<DT><<<grid, 256, 0, st>>>(a, live, live_planes, live_round, batches, rows, cols, shares, (float *)workspace),
         parts_sum_kernel<DT><<<dim3((unsigned)((cols + WAVE - 1) / WAVE), (unsigned)batches), 256, 0, st>>>((const float *)workspace, shares, cols, out)));
    PM_LAUNCH_CHECK(who);
    return 0;
}

extern "C" size_t planmoe_gate_dw_workspace_bytes(int samples, int model_dim, int experts)
{
    if (samples < 1 || model_dim < 1 || experts < 1) return 16;
    return (size_t)reduction_shares(samples, (model_dim + 255) / 256) * experts * model_dim * 4;
}

extern "C" int planmoe_gate_dw(const void *x, int dtype, const float *grad_logits, int samples, int model_dim, int experts, void *out,
                               void *workspace, size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_gate_dw";
    PM_REQUIRE(dtype_ok(dtype) && samples >= 1 && model_dim >= 1 && experts >= 1, "%s: bad shape", who);
    const int vec = dtype == PLANMOE_F32 ? 4 : 8;
    PM_REQUIRE(model_dim % vec == 0 && x && grad_logits && out && aligned16(x), "%s: model_dim must be a multiple of %d, x 16-byte aligned", who, vec);
    PM_REQUIRE(workspace && workspace_bytes >= planmoe_gate_dw_workspace_bytes(samples, model_dim, experts), "%s: workspace too small", who);
    const int shares = reduction_shares(samples, (model_dim + 255) / 256);
    const dim3 grid((unsigned)((model_dim / vec + WAVE - 1) / WAVE), (unsigned)shares);
    hipStream_t st = (hipStream_t)stream;
    for (int e0 = 0; e0 < experts; e0 += 8)
        PM_DTYPE_SWITCH(dtype, DT, (gate_dw_kernel<DT, 8><<<grid, 256, 0, st>>>(x, grad_logits, samples, model_dim, experts, e0, shares, (float *)workspace)));
    PM_DTYPE_SWITCH(dtype, DT, (parts_sum_kernel<DT><<<dim3((unsigned)(((int64_t)experts * model_dim + WAVE - 1) / WAVE), 1u), 256, 0, st>>>(
        (const float *)workspace, shares, experts * model_dim, out)));
    PM_LAUNCH_CHECK(who);
    return 0;
}
