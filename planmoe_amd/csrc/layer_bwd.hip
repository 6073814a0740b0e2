// What the layer's backward pass does besides its products: the bias and gate weight gradients, and the
// gradient of x from the experts' rows and the gate's logits.
//
// A reduction over rows is two stages, shares of the rows and then the sum of the shares.  The first stages of the second
// bias's and the gate weight's gradients share a launch (planmoe_layer_sums), and their last stages the launch that ends the
// first bias's (planmoe_layer_relu_bwd).
#include "layer_rows.hpp"
#include "sums.hpp"

#include <algorithm>

namespace pm {
namespace {

// rows in use of batch e
__device__ __forceinline__ int rows_used(const int *__restrict__ live, int live_planes, int live_round, int batches, int rows, int e)
{
    if (!live) return rows;
    int n = 0;
    for (int j = 0; j < live_planes; ++j) n += live[j * batches + e];
    return min(rows, (n + live_round - 1) / live_round * live_round);
}

// Column sums of the rows in use of every batch: parts[e][share][n] = sum of a[e][r][n] over the share's rows.
// A work-group takes 64 vectors of columns and a share of the rows, four rows at a time side by side.
struct ColsArgs {
    const void *a;
    const int *live;
    int live_planes, live_round, batches, rows, cols, shares, across;      // across: work-groups side by side
    float *parts;
    int blocks() const { return across * shares * batches; }
};
template <int DT>
__device__ __forceinline__ void cols_share(const ColsArgs &p, int block, float *s_sum)
{
    using E = Elem<DT>;
    constexpr int V = E::VEC, LANE = V + 1;
    const int bx = block % p.across, share = block / p.across % p.shares, e = block / p.across / p.shares;
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    const int units = p.cols / V, u = bx * WAVE + lane, uc = min(u, units - 1);
    const int used = rows_used(p.live, p.live_planes, p.live_round, p.batches, p.rows, e);
    const int per = (used + p.shares - 1) / p.shares, r0 = share * per, r1 = min(used, r0 + per);
    const uint4 *src = reinterpret_cast<const uint4 *>((const char *)p.a + (int64_t)e * p.rows * p.cols * (int64_t)sizeof(typename E::store_t));
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
    for (int i = 0; i < V; ++i) s_sum[(wave * WAVE + lane) * LANE + i] = acc[i];
    __syncthreads();
    for (int x = threadIdx.x; x < WAVE * V; x += 256) {
        const int l = x / V, i = x % V, col = (bx * WAVE + l) * V + i;
        auto of = [&](int w) { return s_sum[(w * WAVE + l) * LANE + i]; };
        if (col < p.cols) p.parts[((int64_t)e * p.shares + share) * p.cols + col] = of(0) + of(1) + of(2) + of(3);
    }
}

// Gate weight gradient: parts[share][e][m] = sum_{t in share} g[t][e] * x[t][m]; a work-group takes 64 vectors
// of columns, a share of the tokens, its waves every fourth group of four, and EP experts.
constexpr int GATE_EP = 8;
struct GateArgs {
    const void *x;
    const float *g;
    int samples, model_dim, experts, shares, across;
    float *parts;
    int blocks() const { return across * shares * ((experts + GATE_EP - 1) / GATE_EP); }
};
template <int DT>
__device__ __forceinline__ void gate_share(const GateArgs &p, int block, float *s_sum)
{
    using E = Elem<DT>;
    constexpr int V = E::VEC, EP = GATE_EP, LANE = EP * V + 1;
    const int bx = block % p.across, share = block / p.across % p.shares, e0 = block / p.across / p.shares * EP;
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int units = p.model_dim / V, u = bx * WAVE + lane, uc = min(u, units - 1);
    const int per = (p.samples + p.shares - 1) / p.shares, t0 = share * per, t1 = min(p.samples, t0 + per);
    const uint4 *src = reinterpret_cast<const uint4 *>(p.x);
    float acc[EP][V];
#pragma unroll
    for (int e = 0; e < EP; ++e)
#pragma unroll
        for (int i = 0; i < V; ++i) acc[e][i] = 0.f;
    constexpr int R = 4;
    for (int t = t0 + wave * R; t < t1; t += 4 * R) {
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
                const float ge = e0 + e < p.experts && t + q < t1 ? E::round(p.g[(int64_t)tq * p.experts + e0 + e]) : 0.f;
#pragma unroll
                for (int i = 0; i < V; ++i) acc[e][i] = fmaf(ge, f[i], acc[e][i]);
            }
        }
    }
    if (wave > 0)
#pragma unroll
        for (int e = 0; e < EP; ++e)
#pragma unroll
            for (int i = 0; i < V; ++i) s_sum[((wave - 1) * WAVE + lane) * LANE + e * V + i] = acc[e][i];
    __syncthreads();
    if (wave == 0 && u < units) {
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            if (e0 + e >= p.experts) break;
            float *to = p.parts + ((int64_t)share * p.experts + e0 + e) * p.model_dim + (int64_t)u * V;
#pragma unroll
            for (int i = 0; i < V; ++i) {
                auto of = [&](int w) { return s_sum[(w * WAVE + lane) * LANE + e * V + i]; };
                to[i] = acc[e][i] + of(0) + of(1) + of(2);
            }
        }
    }
}

// the first stages of either or both (the work-groups of the column sums come first)
template <int DT, bool COLS, bool GATE>
__global__ __launch_bounds__(256) void shares_kernel(const ColsArgs cols, const GateArgs gate, int col_blocks)
{
    constexpr int V = Elem<DT>::VEC, FOR_COLS = 4 * WAVE * (V + 1), FOR_GATE = 3 * WAVE * (GATE_EP * V + 1);
    __shared__ float s_sum[GATE ? std::max(FOR_GATE, FOR_COLS) : FOR_COLS];
    const int b = (int)blockIdx.x;
    if constexpr (COLS) {
        if (!GATE || b < col_blocks) { cols_share<DT>(cols, b, s_sum); return; }
    }
    if constexpr (GATE) gate_share<DT>(gate, b - col_blocks, s_sum);
}

// the slots' sums of up to SUM_JOBS reductions: 64 columns per work-group, its waves every fourth eight slots, eight loads in flight
// (a thread per column that walked the slots one by one took 35 us for 256 slots of 8 x 1024)
struct SumJobs { SumJob job[SUM_JOBS]; int first[SUM_JOBS]; };
template <int DT>
__global__ __launch_bounds__(256) void slots_sum_kernel(const SumJobs all)
{
    __shared__ float s_sum[4][WAVE];
    int which = 0, b = (int)blockIdx.x;
#pragma unroll
    for (int i = 1; i < SUM_JOBS; ++i) if (b >= all.first[i]) which = i;
    const SumJob p = all.job[which];
    b -= all.first[which];
    const int across = (p.cols + WAVE - 1) / WAVE, e = b / across, lane = lane_id(), wave = threadIdx.x >> 6, c = (b - e * across) * WAVE + lane;
    int used = p.slots;
    if (p.live) {
        const int rows = rows_used(p.live, p.live_planes, p.live_round, p.batches, p.rows, e);
        used = min(used, (rows + p.slot_rows - 1) / p.slot_rows * p.per_tile);
    }
    const float *from = p.from + (int64_t)e * p.slots * p.cols + min(c, p.cols - 1);
    float s = 0.f;
    for (int i = wave * 8; i < used; i += 32) {
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = from[(int64_t)min(i + q, used - 1) * p.cols];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = i + q < used ? v[q] : 0.f;
        // (in pairs: up to eight slots are one wave's, and one after the other are seven roundings of the whole sum)
        s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    s_sum[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && c < p.cols) Elem<DT>::store(p.out, (int64_t)e * p.cols + c, s_sum[0][lane] + s_sum[1][lane] + s_sum[2][lane] + s_sum[3][lane]);
}

// out[t] = round(sum_j codec(rows[slot_j])) + sum_e g[t][e] * wg[e]: the combine of the gradient rows and the gate's share of the
// gradient of x in one pass (their own launches read and write out once more).  A wave per TOKENS tokens; up to EP experts, whose
// weights come from the caches.  The roundings are those of planmoe_layer_combine and planmoe_gate_dx_accumulate.  Bound by the rows' bytes and, for
// wide rows, by the weights out of L2.  bf16, top-2, 8 experts, both launches and this one: 16384 x 1024 44 and 24 us (int8 46 and 34), x 4096
// 141 and 100 (int8 145 and 127), 1024 x 1024 17 and 7.5.  (Up to 16 experts: where it pays, by dx_in_one of ext/layer.cpp.)
template <int DT, int CACHE, bool INT8, int EP, int TOKENS>
__global__ __launch_bounds__(256) void layer_dx_kernel(
    const void *__restrict__ rows, const int32_t *__restrict__ indices, const int32_t *__restrict__ locations, int64_t stride, int top_k,
    int samples, int model_dim, int capacity, const float *__restrict__ g, const void *__restrict__ wg, int experts, void *__restrict__ out)
{
    using E = Elem<DT>;
    constexpr int V = E::VEC;
    __shared__ __align__(16) float s_table[INT8 ? 4 : 1][256];
    const int lane = lane_id(), units = model_dim / V;
    const int t0 = __builtin_amdgcn_readfirstlane((blockIdx.x * 4 + (threadIdx.x >> 6)) * TOKENS);
    if (t0 >= samples) return;                   // (no work-group barrier below)
    float *const table = s_table[INT8 ? threadIdx.x >> 6 : 0];
    float acc[TOKENS][CACHE][V];
#pragma unroll
    for (int k = 0; k < TOKENS; ++k) {
        const int t = min(t0 + k, samples - 1);
        for (int j0 = 0; j0 < top_k; j0 += WAVE) {
            const int np = min(top_k - j0, WAVE);
            int slot; float gate;
            fetch_planes(nullptr, indices, locations, stride, t, j0, np, 0x7fffffff, capacity, slot, gate);
            // the next choice's row is on its way while this one's is worked on (a dropped choice reads slot 0, unused)
            uint4 next[CACHE];
            auto request = [&](int j) {
                const uint4 *src = reinterpret_cast<const uint4 *>(rows) + (int64_t)max(rl_i(slot, j), 0) * units;
#pragma unroll
                for (int c = 0; c < CACHE; ++c) next[c] = src[min(c * WAVE + lane, units - 1)];
            };
            request(0);
            for (int j = 0; j < np; ++j) {
                const int s = rl_i(slot, j);
                uint4 row[CACHE];
#pragma unroll
                for (int c = 0; c < CACHE; ++c) row[c] = next[c];
                if (j + 1 < np) request(j + 1);
                auto add = [&](int c, const float (&f)[V]) {
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        const float v = s >= 0 ? f[i] : 0.f;
                        acc[k][c][i] = j0 + j == 0 ? v : acc[k][c][i] + v;
                    }
                };
                if constexpr (INT8) {
                    const RowTable<DT> tab(row, 1.f, table);
                    table_sync();
                    auto body = [&](auto mode) {
#pragma unroll
                        for (int c = 0; c < CACHE; ++c) {
                            float f[V];
                            tab.template values<decltype(mode)::value>(row[c], f);
                            add(c, f);
                        }
                    };
                    if (tab.enc.fast()) body(std::true_type{}); else body(std::false_type{});
                    table_sync();                // (the next choice's table takes this one's place)
                } else {
#pragma unroll
                    for (int c = 0; c < CACHE; ++c) {
                        float f[V];
                        E::unpack(row[c], f);
                        add(c, f);
                    }
                }
            }
        }
    }
    float ge[TOKENS][EP];
#pragma unroll
    for (int k = 0; k < TOKENS; ++k)
#pragma unroll
        for (int e = 0; e < EP; ++e)
            ge[k][e] = E::round(g[(int64_t)min(t0 + k, samples - 1) * experts + min(e, experts - 1)]);
    uint4 *dst = reinterpret_cast<uint4 *>(out) + (int64_t)t0 * units;
    const uint4 *weights = reinterpret_cast<const uint4 *>(wg);
#pragma unroll
    for (int c = 0; c < CACHE; ++c) {
        const int u = c * WAVE + lane;
#pragma unroll
        for (int k = 0; k < TOKENS; ++k)
#pragma unroll
            for (int i = 0; i < V; ++i) acc[k][c][i] = E::round(acc[k][c][i]);
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            float w[V];
            E::unpack(weights[(int64_t)min(e, experts - 1) * units + min(u, units - 1)], w);
#pragma unroll
            for (int k = 0; k < TOKENS; ++k)
#pragma unroll
                for (int i = 0; i < V; ++i) acc[k][c][i] = e < experts ? fmaf(ge[k][e], w[i], acc[k][c][i]) : acc[k][c][i];
        }
#pragma unroll
        for (int k = 0; k < TOKENS; ++k)
            if (u < units && t0 + k < samples) stream_store(dst + (int64_t)k * units + u, E::pack(acc[k][c]));
    }
}

// The same for few tokens, bound by trips to memory one after the other: the waves of a work-group share a token's row, PER vectors a lane each, and what
// does not depend on the slots, the weights above all, is asked for before them (layer_dx_kernel asks for EP vectors, then the next EP, behind the
// rows).  With the codec every wave reads the whole row, whose minimum and scale it needs.  The same operations in the same order.  us, layer_dx_kernel
// and this one, two choices of 8 experts, 5, 300, 1500 and 3000 tokens:
//   fp32        x 920  9.0, 3.2   11.7, 4.2   14.6, 7.1    16.7, 10.3      x 2048  16.2, 3.6   21.4, 5.2   27.0, 11.3   29.1, 17.3
//   fp32, int8  x 768  10.4, 5.0  12.6, 6.1   15.0, 12.1   16.8, 19.1      bf16, int8  x 4096  12.4, 6.2  13.5, 9.1  19.5, 21.9  31.0, 39.8
template <int DT, int CACHE, bool INT8, int EP>
__global__ __launch_bounds__(256) void layer_dx_few_kernel(
    const void *__restrict__ rows, const int32_t *__restrict__ indices, const int32_t *__restrict__ locations, int64_t stride, int top_k,
    int samples, int model_dim, int capacity, const float *__restrict__ g, const void *__restrict__ wg, int experts, void *__restrict__ out)
{
    using E = Elem<DT>;
    constexpr int V = E::VEC, PER = CACHE > 4 ? CACHE / 4 : 1, ACROSS = CACHE / PER;       // vectors of a wave, waves of a token
    __shared__ __align__(16) float s_table[INT8 ? 4 : 1][256];
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), units = model_dim / V;
    const int t = blockIdx.x * (4 / ACROSS) + wave / ACROSS, c0 = wave % ACROSS * PER;
    if (t >= samples) return;                    // (no work-group barrier below)
    float *const table = s_table[INT8 ? wave : 0];
    auto unit = [&](int c) { return min((c0 + c) * WAVE + lane, units - 1); };
    uint4 weight[EP][PER];
    float ge[EP];
#pragma unroll
    for (int e = 0; e < EP; ++e) {
        ge[e] = g[(int64_t)t * experts + min(e, experts - 1)];
#pragma unroll
        for (int c = 0; c < PER; ++c) weight[e][c] = reinterpret_cast<const uint4 *>(wg)[(int64_t)min(e, experts - 1) * units + unit(c)];
    }
    float acc[PER][V];
    for (int j0 = 0; j0 < top_k; j0 += WAVE) {
        const int np = min(top_k - j0, WAVE);
        int slot; float gate;
        fetch_planes(nullptr, indices, locations, stride, t, j0, np, 0x7fffffff, capacity, slot, gate);
        // the next choice's row is on its way while this one's is worked on (a dropped choice reads slot 0, unused)
        uint4 next[PER], all[INT8 ? CACHE : 1];       // (a wave that has the whole row has it once)
        auto request = [&](int j) {
            const uint4 *src = reinterpret_cast<const uint4 *>(rows) + (int64_t)max(rl_i(slot, j), 0) * units;
            if constexpr (!INT8 || ACROSS > 1)
#pragma unroll
                for (int c = 0; c < PER; ++c) next[c] = src[unit(c)];
            if constexpr (INT8)
#pragma unroll
                for (int c = 0; c < CACHE; ++c) all[c] = src[min(c * WAVE + lane, units - 1)];
        };
        request(0);
        for (int j = 0; j < np; ++j) {
            const int s = rl_i(slot, j);
            uint4 row[PER], whole[INT8 ? CACHE : 1];
#pragma unroll
            for (int c = 0; c < PER; ++c) row[c] = INT8 && ACROSS == 1 ? all[c] : next[c];
            if constexpr (INT8)
#pragma unroll
                for (int c = 0; c < CACHE; ++c) whole[c] = all[c];
            if (j + 1 < np) request(j + 1);
            auto add = [&](int c, const float (&f)[V]) {
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const float v = s >= 0 ? f[i] : 0.f;
                    acc[c][i] = j0 + j == 0 ? v : acc[c][i] + v;
                }
            };
            if constexpr (INT8) {
                const RowTable<DT> tab(whole, 1.f, table);
                table_sync();
                auto body = [&](auto mode) {
#pragma unroll
                    for (int c = 0; c < PER; ++c) {
                        float f[V];
                        tab.template values<decltype(mode)::value>(row[c], f);
                        add(c, f);
                    }
                };
                if (tab.enc.fast()) body(std::true_type{}); else body(std::false_type{});
                table_sync();                    // (the next choice's table takes this one's place)
            } else {
#pragma unroll
                for (int c = 0; c < PER; ++c) {
                    float f[V];
                    E::unpack(row[c], f);
                    add(c, f);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < PER; ++c) {
#pragma unroll
        for (int i = 0; i < V; ++i) acc[c][i] = E::round(acc[c][i]);
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            const float scale = E::round(ge[e]);
            float w[V];
            E::unpack(weight[e][c], w);
#pragma unroll
            for (int i = 0; i < V; ++i) acc[c][i] = e < experts ? fmaf(scale, w[i], acc[c][i]) : acc[c][i];
        }
        const int u = (c0 + c) * WAVE + lane;
        if (u < units) stream_store(reinterpret_cast<uint4 *>(out) + (int64_t)t * units + u, E::pack(acc[c]));
    }
}

// how many shares a reduction over `rows` is cut into for `blocks` column blocks: enough work-groups for the GPU, at least 32 rows each
int reduction_shares(int64_t rows, int64_t blocks)
{
    int64_t s = (1024 + blocks - 1) / blocks;
    if (s > (rows + 31) / 32) s = (rows + 31) / 32;
    return (int)(s < 1 ? 1 : s > 256 ? 256 : s);
}

ColsArgs cols_args(const void *a, int dtype, int batches, int rows, int cols, const int32_t *live, int live_planes, int live_round, void *parts)
{
    const int vec = dtype == PLANMOE_F32 ? 4 : 8;
    return ColsArgs{a, live, live_planes, live_round, batches, rows, cols, reduction_shares(rows, (int64_t)batches * ((cols + 255) / 256)),
                    (cols / vec + WAVE - 1) / WAVE, (float *)parts};
}
GateArgs gate_args(const void *x, int dtype, const float *g, int samples, int model_dim, int experts, void *parts)
{
    const int vec = dtype == PLANMOE_F32 ? 4 : 8;
    return GateArgs{x, g, samples, model_dim, experts, reduction_shares(samples, (model_dim + 255) / 256), (model_dim / vec + WAVE - 1) / WAVE, (float *)parts};
}
SumJob sum_of(const ColsArgs &p, void *out) { return SumJob{p.parts, out, p.batches, p.shares, p.cols, nullptr, 1, 1, 0, 1, 1}; }
SumJob sum_of(const GateArgs &p, void *out) { return SumJob{p.parts, out, 1, p.shares, p.experts * p.model_dim, nullptr, 1, 1, 0, 1, 1}; }

int check_cols(const char *who, const void *a, int dtype, int batches, int rows, int cols, const int32_t *live, int live_planes, int live_round)
{
    PM_REQUIRE(dtype_ok(dtype) && batches >= 1 && rows >= 1 && cols >= 1, "%s: bad shape", who);
    const int vec = dtype == PLANMOE_F32 ? 4 : 8;
    PM_REQUIRE(cols % vec == 0 && a && aligned16(a), "%s: cols must be a multiple of %d, the rows 16-byte aligned", who, vec);
    PM_REQUIRE(batches < 65536 && (!live || (live_planes >= 1 && live_round >= 1)), "%s: bad live rows", who);
    return 0;
}
int check_gate(const char *who, const void *x, int dtype, const float *grad_logits, int samples, int model_dim, int experts)
{
    PM_REQUIRE(dtype_ok(dtype) && samples >= 1 && model_dim >= 1 && experts >= 1, "%s: bad shape", who);
    const int vec = dtype == PLANMOE_F32 ? 4 : 8;
    PM_REQUIRE(model_dim % vec == 0 && x && grad_logits && aligned16(x), "%s: model_dim must be a multiple of %d, x 16-byte aligned", who, vec);
    PM_REQUIRE((int64_t)experts * model_dim < (1ll << 31), "%s: too many weights", who);
    return 0;
}

} // namespace

int sum_slots(const char *who, int dtype, const SumJob *jobs, int n, hipStream_t st)
{
    SumJobs all{};
    int64_t blocks = 0;
    for (int i = 0; i < SUM_JOBS; ++i) {
        if (i < n) all.job[i] = jobs[i];
        all.first[i] = i == 0 ? 0 : i < n ? (int)blocks : 0x7fffffff;
        if (i < n) blocks += (int64_t)jobs[i].batches * ((jobs[i].cols + WAVE - 1) / WAVE);
        PM_REQUIRE(blocks < (1ll << 31), "%s: too many columns", who);
    }
    if (blocks == 0) return 0;
    PM_DTYPE_SWITCH(dtype, DT, (slots_sum_kernel<DT><<<(unsigned)blocks, 256, 0, st>>>(all)));
    PM_LAUNCH_CHECK(who);
    return 0;
}

} // namespace pm

using namespace pm;

extern "C" size_t planmoe_rows_colsum_workspace_bytes(int batches, int rows, int cols)
{
    if (batches < 1 || rows < 1 || cols < 1) return 16;
    return (size_t)batches * reduction_shares(rows, (int64_t)batches * ((cols + 255) / 256)) * cols * 4;
}

extern "C" int planmoe_rows_colsum(const void *a, int dtype, int batches, int rows, int cols, const int32_t *live, int live_planes,
                                   int live_round, void *out, void *workspace, size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_rows_colsum";
    if (check_cols(who, a, dtype, batches, rows, cols, live, live_planes, live_round)) return 1;
    PM_REQUIRE(out && workspace && workspace_bytes >= planmoe_rows_colsum_workspace_bytes(batches, rows, cols), "%s: NULL output, or workspace too small", who);
    hipStream_t st = (hipStream_t)stream;
    const ColsArgs p = cols_args(a, dtype, batches, rows, cols, live, live_planes, live_round, workspace);
    PM_DTYPE_SWITCH(dtype, DT, (shares_kernel<DT, true, false><<<p.blocks(), 256, 0, st>>>(p, GateArgs{}, p.blocks())));
    const SumJob last = sum_of(p, out);
    return sum_slots(who, dtype, &last, 1, st);
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
    if (check_gate(who, x, dtype, grad_logits, samples, model_dim, experts)) return 1;
    PM_REQUIRE(out && workspace && workspace_bytes >= planmoe_gate_dw_workspace_bytes(samples, model_dim, experts), "%s: NULL output, or workspace too small", who);
    hipStream_t st = (hipStream_t)stream;
    const GateArgs p = gate_args(x, dtype, grad_logits, samples, model_dim, experts, workspace);
    PM_DTYPE_SWITCH(dtype, DT, (shares_kernel<DT, false, true><<<p.blocks(), 256, 0, st>>>(ColsArgs{}, p, 0)));
    const SumJob last = sum_of(p, out);
    return sum_slots(who, dtype, &last, 1, st);
}

static size_t cols_bytes(int batches, int rows, int cols) { return round_up(planmoe_rows_colsum_workspace_bytes(batches, rows, cols), 256); }

extern "C" size_t planmoe_layer_sums_workspace_bytes(int experts, int capacity, int samples, int model_dim)
{
    return cols_bytes(experts, capacity, model_dim) + planmoe_gate_dw_workspace_bytes(samples, model_dim, experts);
}

extern "C" int planmoe_layer_sums(const void *grad_rows, int dtype, int experts, int capacity, const int32_t *live, int live_planes,
                                  int live_round, const void *x, const float *grad_logits, int samples, int model_dim, void *workspace,
                                  size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_layer_sums";
    if (check_cols(who, grad_rows, dtype, experts, capacity, model_dim, live, live_planes, live_round)) return 1;
    if (check_gate(who, x, dtype, grad_logits, samples, model_dim, experts)) return 1;
    PM_REQUIRE(workspace && workspace_bytes >= planmoe_layer_sums_workspace_bytes(experts, capacity, samples, model_dim), "%s: workspace too small", who);
    const ColsArgs cols = cols_args(grad_rows, dtype, experts, capacity, model_dim, live, live_planes, live_round, workspace);
    const GateArgs gate = gate_args(x, dtype, grad_logits, samples, model_dim, experts, (char *)workspace + cols_bytes(experts, capacity, model_dim));
    PM_DTYPE_SWITCH(dtype, DT, (shares_kernel<DT, true, true><<<cols.blocks() + gate.blocks(), 256, 0, (hipStream_t)stream>>>(cols, gate, cols.blocks())));
    PM_LAUNCH_CHECK(who);
    return 0;
}

extern "C" int planmoe_layer_relu_bwd(int dtype, const void *grad_rows, const void *w2, const void *h, int experts, int capacity, int hidden,
                                      int model_dim, const int32_t *live, int live_planes, int live_round, int rows_hint, void *grad_h,
                                      void *db1, void *workspace, size_t workspace_bytes, const void *sums, size_t sums_bytes, int samples,
                                      void *db2, void *dwg, void *stream)
{
    const char *who = "planmoe_layer_relu_bwd";
    PM_REQUIRE(experts >= 1 && capacity >= 1 && samples >= 1 && model_dim >= 1 && db1 && db2 && dwg, "%s: bad shape or NULL output", who);
    PM_REQUIRE(sums && sums_bytes >= planmoe_layer_sums_workspace_bytes(experts, capacity, samples, model_dim), "%s: sums too small", who);
    void *parts = const_cast<void *>(sums);
    const SumJob others[2] = {sum_of(cols_args(nullptr, dtype, experts, capacity, model_dim, live, live_planes, live_round, parts), db2),
                              sum_of(gate_args(nullptr, dtype, nullptr, samples, model_dim, experts, (char *)parts + cols_bytes(experts, capacity, model_dim)), dwg)};
    return relu_bwd_with(who, dtype, grad_rows, w2, h, experts, capacity, hidden, model_dim, live, live_planes, live_round, rows_hint, grad_h, db1, workspace,
                         workspace_bytes, others, 2, (hipStream_t)stream);
}

// Up to how many tokens layer_dx_few_kernel takes less than layer_dx_kernel (for rows above 8 KB than the two launches), whose trips other waves hide beyond.
// Time of the first by that of the second, means over row lengths, one choice and two, 7 experts and 12 and 16, at so many tokens:
//   vectors a lane, fp32 (7)                  16 bits (7)                               fp32 (12, 16)              16 bits (12, 16)
//   1                1000 0.84   4000 0.85    1000 0.97   1400 1.02                     2000 0.89   2800 1.00      60 1.05   1000 1.02
//   2 to 4           1000 0.69   4000 0.72    1000 0.93   1400 0.95   2000 1.04         1400 0.85   2000 0.96      1000 0.94   1400 0.98   2000 1.12
//   5 to 8           1000 0.50   4000 0.68    1000 0.88   1400 0.90   2000 1.05         1400 0.94   2000 1.17      767 0.91   1000 1.06
//   9 to 16          1000 0.56   4000 0.85    1000 0.54   2800 0.82   4000 0.93 (12 KB, 3 and 4 experts 1.07)
// and through the codec, where every wave reads the whole row
//   1                500 0.87   767 0.87      500 0.98   767 0.97                       500 0.71   767 0.71        60 1.04   767 1.01
//   2 to 4           500 0.67   767 0.76      500 0.82   767 0.99                       500 0.56   767 0.65        500 0.79   767 0.97
//   5 to 8           500 0.51   767 0.74      500 0.75   767 0.99                       500 0.50   767 0.72        500 0.92   767 1.29
//   9 to 16 (beyond 256 fp32 x 4096 25.7 us at 700 tokens, 34.2 so)   60 0.48           16 bits 60 0.39
static int64_t dx_few_tokens(int dtype, int codec, int per_lane, int experts)
{
    const bool f32 = dtype == PLANMOE_F32, many = experts > 8;
    int64_t a_unit;                              // tokens a compute unit
    if (!f32 && many && per_lane == 1) a_unit = 0;
    else if (codec) a_unit = per_lane > 8 ? 1 : f32 ? 3 : 2;
    else if (f32) a_unit = !many ? 16 : per_lane > 2 ? 6 : 8;
    else a_unit = per_lane > 8 ? 12 : per_lane > 4 ? many ? 3 : 6 : per_lane > 1 ? 5 : 4;
    return a_unit * compute_units();
}

extern "C" int planmoe_layer_dx(const void *rows, int dtype, int codec, const int32_t *indices, const int32_t *locations, int64_t plane_stride,
                                int top_k, int samples, int model_dim, int experts, int capacity, const float *grad_logits, const void *wg,
                                void *out, void *stream)
{
    const char *who = "planmoe_layer_dx";
    if (layer_rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, codec)) return 1;
    PM_REQUIRE(experts <= 16, "%s: built for up to 16 experts (got %d)", who, experts);
    if (samples == 0) return 0;
    PM_REQUIRE(grad_logits && wg && out && aligned16(wg) && aligned16(out), "%s: NULL or unaligned argument", who);
    const int per_lane = (model_dim / (dtype == PLANMOE_F32 ? 4 : 8) + WAVE - 1) / WAVE;
    PM_REQUIRE(experts <= 8 || per_lane <= 8, "%s: more than 8 experts: rows of up to 8 KB", who);
    const bool few = samples <= dx_few_tokens(dtype, codec, per_lane, experts);
    if (per_lane > 8 && !few) {
        if (planmoe_layer_combine(rows, dtype, codec, nullptr, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, out, stream)) return 1;
        return planmoe_gate_dx_accumulate(out, dtype, grad_logits, wg, samples, model_dim, experts, stream);
    }
    hipStream_t st = (hipStream_t)stream;
    // Two tokens a wave read the weights once where they are as wide as the cache they come from and there are waves enough
    // (fp32, 8 experts x 1024 x 16384 tokens, no codec: 69 us with one, 34 with two; x 1024 tokens: 7.3 and 6.0, int8 10.1 and 11.4; bf16, whose rows
    // take twice the registers unpacked: 43 and 39, int8 59 and 61).  16 experts' weights at any number of tokens that is not few.
    const bool pairs = dtype == PLANMOE_F32 && (samples >= 4096 || experts > 8);
#define PM_DX__(CACHE, INT8, EP, TOKENS) (layer_dx_kernel<DT, CACHE, INT8, EP, TOKENS><<<(samples + 4 * TOKENS - 1) / (4 * TOKENS), 256, 0, st>>>( \
        rows, indices, locations, plane_stride, top_k, samples, model_dim, capacity, grad_logits, wg, experts, out))
#define PM_DX_FEW(CACHE, INT8, EP)                                                                              \
    do {                                                                                                        \
        constexpr int TOKENS = CACHE >= 4 ? 1 : 4 / CACHE;                                                      \
        layer_dx_few_kernel<DT, CACHE, INT8, EP><<<(samples + TOKENS - 1) / TOKENS, 256, 0, st>>>(              \
            rows, indices, locations, plane_stride, top_k, samples, model_dim, capacity, grad_logits, wg, experts, out);            \
    } while (0)
#define PM_DX_(CACHE, INT8, EP)                                                                                 \
    do {                                                                                                        \
        if constexpr (DT == PLANMOE_F32 || EP <= 8 || CACHE > 1) { if (few) { PM_DX_FEW(CACHE, INT8, EP); break; } }                \
        if constexpr (DT == PLANMOE_F32) { if (pairs) { PM_DX__(CACHE, INT8, EP, 2); break; } }                 \
        PM_DX__(CACHE, INT8, EP, 1);                                                                            \
    } while (0)
#define PM_DX(CACHE)                                                                                            \
    do {                                                                                                        \
        if (codec) { if (experts <= 4) PM_DX_(CACHE, true, 4); else if (experts <= 8) PM_DX_(CACHE, true, 8); else PM_DX_(CACHE, true, 16); }      \
        else { if (experts <= 4) PM_DX_(CACHE, false, 4); else if (experts <= 8) PM_DX_(CACHE, false, 8); else PM_DX_(CACHE, false, 16); }         \
    } while (0)
#define PM_DX_WIDE() do { if (codec) PM_DX_FEW(16, true, 8); else PM_DX_FEW(16, false, 8); } while (0)
    PM_DTYPE_SWITCH(dtype, DT, { if (per_lane <= 1) PM_DX(1); else if (per_lane <= 2) PM_DX(2); else if (per_lane <= 4) PM_DX(4); else if (per_lane <= 8) PM_DX(8); else PM_DX_WIDE(); });
#undef PM_DX_WIDE
#undef PM_DX_FEW
#undef PM_DX
#undef PM_DX_
#undef PM_DX__
    PM_LAUNCH_CHECK(who);
    return 0;
}
