// The layer's first product for few tokens (decode), which routes them itself.
//
// A decode step reads its weights once; before that the gate's launch takes 8 us of one work-group's latencies (8 tokens x 1024: launch,
// loads, products, softmax, ranks, one after the other) while memory has nothing to do.  Here every work-group of the first product
// (gemm_skinny.hip) routes all tokens for itself: four of its sixteen waves are the gate's work-group (gate_route.hpp; x and the gate's
// weight come from L2), the other twelve have asked for their share of the expert's weight before they wait for them.  A work-group then knows
// its expert's tokens and takes their rows straight from x, through the int8 codec where the exchange has one, so that
// the dispatched rows are neither written nor read.  Same roundings and the same order of sums as the launches it stands for.
//
// Bound by reading the weights and the gate's latency under it.  us in two launches and in one, without a codec and through it, weights in the last cache
// (where they fit) and cold, 4 experts top-1, 8 and 16 top-2:
//   1 token     4, 4096 -> 512   18.3, 11.9 and 20.0, 18.0   21.8, 21.1 and 22.4, 20.0      8, 1024 -> 4096  14.6, 13.1 and 15.2, 13.7   15.2, 15.0 and 16.0, 15.6
//               8, 2048 -> 4096  23.1, 21.1 and 23.9, 22.8   23.6, 23.2 and 24.3, 24.5
//   8 tokens    8, 256 -> 512    8.4, 6.3 and 8.8, 6.9       8.8, 6.6 and 9.2, 7.2          8, 1024 -> 4096  18.8, 15.6 and 18.9, 16.2   20.1, 17.0 and 20.9, 17.5
//   32 tokens   8, 4096 -> 512   29.9, 23.1 and 31.7, 27.1   37.7, 30.8 and 39.3, 32.0      8, 4096 -> 4096  60.7, 54.5 and 62.1, 55.4   60.0, 54.9 and 61.8, 55.9
//               16, 4096 -> 2048 63.2, 56.4 and 63.8, 57.2   62.7, 57.0 and 64.4, 57.7      4, 4096 -> 2048  30.1, 23.1 and 31.8, 26.4   37.3, 30.1 and 39.0, 31.5
// (190 shapes of 1, 8 and 32 tokens, 256 to 4096 -> 512 to 4096: 0.84 of two launches, at worst 1.03)
#include "gate_route.hpp"
#include "gemm_shares.hpp"
#include "gemm_skinny_core.hpp"

namespace pm {

struct FirstArgs {
    const void *x, *wg;
    int samples, top_k, normalize_gate;
    int32_t *indices, *locations;
    void *gates;
    int64_t stride;
    float *l_aux;
    int32_t *counts;
};

constexpr int FIRST_WAVES = 16, FIRST_TOKENS = 32, FIRST_ROWS = 16;          // a group's tokens, an expert's rows

// TOKENS: a group's, 16 or 32.  CAP: bound of the number of experts.  DECODED: rows go through the int8 codec.  C, U, LARGE: as gemm_skinny_kernel
template <int TOKENS, int CAP, bool DECODED, int C, int U, bool LARGE>
__global__ __launch_bounds__(FIRST_WAVES * 64) void layer_first_kernel(const SkinnyArgs p, const FirstArgs r)
{
    constexpr int ONE = DECODED ? OUT_DECODED : OUT_ROWS;
    extern __shared__ __align__(16) float part[];           // [FIRST_WAVES][16][16 C + 4]
    __shared__ GateShared<PLANMOE_BF16, 1, CAP, true, TOKENS, 0, ONE> sh;
    __shared__ int32_t s_token[FIRST_ROWS];                 // the expert's rows
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int e, n0;
    skinny_tile<16 * C, C == 2>(e, n0);
    const __amdgpu_buffer_rsrc_t da = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(r.x), 0, r.samples * p.K * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(p.B + (int64_t)e * p.N * p.K), 0, (int)((int64_t)p.N * p.K * 2), 0x00020000);
    const int l16 = lane & 15, g = lane >> 4, steps = (p.K + 31) / 32;
    const uint32_t place = n0 + C * l16 < p.N ? ((uint32_t)(8 * g) * (uint32_t)p.N + (uint32_t)(n0 + C * l16)) * 2u : SK_NOWHERE;

    SkinnyWeights<C, LARGE> b[U];
    auto ask = [&] {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (wave + u * FIRST_WAVES < steps) b[u].load(db, place, wave + u * FIRST_WAVES, p.N);
    };
    if (wave < 4) {
        const bool first = blockIdx.x == 0 && blockIdx.y == 0;
        // (16 tokens with four steps on their way, as the gate's launch has them, are more registers than these waves have: 16 x 3840 -> 256, 8 tokens, a pass
        // of the layer 36.8 us, with two 32.8)
        gate_route_group<PLANMOE_BF16, PLANMOE_F32, 1, CAP, true, TOKENS, 0, ONE, 2>(sh, first, 0, 1, r.x, r.wg, nullptr, r.samples, p.K, p.batches, r.top_k,
            r.normalize_gate, r.indices, r.locations, r.gates, r.stride, nullptr, nullptr, first ? r.l_aux : nullptr, r.counts, nullptr, p.M);
        if (wave == 0) {                                    // (the wave that wrote the slots)
            __builtin_amdgcn_wave_barrier();
            for (int j = 0; j < r.top_k; ++j) {
                const int at = lane < TOKENS ? sh.slot[j][lane] - e * p.M : -1;        // (-1 becomes negative: no slot)
                if (at >= 0 && at < p.M) s_token[at] = lane;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        ask();
    } else {
        ask();
        // (as many barriers as the gate's waves meet at; what has been asked for stays on its way)
        asm volatile("s_barrier\n\ts_barrier\n\ts_barrier" ::: "memory");
    }
    const int rows = min(p.M, __builtin_amdgcn_readfirstlane(sh.total[e]));
    if (rows == 0) return;

    // a lane's row of x, and what the codec makes of its values
    const int token = l16 < rows ? s_token[l16] : -1;
    const uint32_t at = token >= 0 ? ((uint32_t)token * (uint32_t)p.K + 8u * (uint32_t)g) * 2u : SK_NOWHERE;
    float mn = 0.f, mx = 0.f;
    if constexpr (DECODED) { mn = sh.range[max(token, 0)][0]; mx = sh.range[max(token, 0)][1]; }
    const float scale = Elem<PLANMOE_BF16>::round(mx - mn);
    const RowEncoder<PLANMOE_BF16> enc(mn, scale);
    const RowDecoder<PLANMOE_BF16> dec(mn, scale);
    const bool fast = __ballot(token >= 0 && !enc.rq.fast) == 0;        // (the wave's rows: what is right for all of them)
    auto through_codec = [&](const pm_u32x4 &a, int step) {
        if constexpr (!DECODED) return a;
        const uint4 raw = make_uint4(a.x, a.y, a.z, a.w);
        uint32_t w[2];
        if (fast) enc.encode<true>(raw, w); else enc.encode<false>(raw, w);
        float f[8];
        dec.word(w[0], f);
        dec.word(w[1], f + 4);
        const uint4 v = Elem<PLANMOE_BF16>::pack(f);
        // (what is no row, or behind a row's end, stays zero: a code of zero is the row's minimum)
        return token >= 0 && step * 32 + 8 * g < p.K ? pm_u32x4{v.x, v.y, v.z, v.w} : pm_u32x4{0u, 0u, 0u, 0u};
    };
    pm_u32x4 a[U][1];
    auto ask_rows = [&](int u, int s) { a[u][0] = __builtin_amdgcn_raw_buffer_load_b128(da, s * 32 + 8 * g < p.K ? at : SK_NOWHERE, (uint32_t)s * 64u, 0); };
    f32x4 acc[1][C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[0][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (wave + u * FIRST_WAVES < steps) ask_rows(u, wave + u * FIRST_WAVES);
    for (int s0 = wave; s0 < steps; s0 += U * FIRST_WAVES) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = s0 + u * FIRST_WAVES, next = s + U * FIRST_WAVES;
            if (s < steps) {
                const pm_u32x4 v[1] = {through_codec(a[u][0], s)};
                b[u].multiply(v, acc);
            }
            if (next < steps) {
                b[u].load(db, place, next, p.N);
                ask_rows(u, next);
            }
        }
    }
    skinny_finish<false, 1, C, FIRST_WAVES, false>(p, e, n0, rows, acc, part);
}

template <int TOKENS, int CAP, bool DECODED, int C, int U, bool LARGE>
static int first_launch(const SkinnyArgs &p, const FirstArgs &r, hipStream_t stream, const char *who)
{
    constexpr int COLS = 16 * C, LDS = FIRST_WAVES * 16 * (COLS + 4) * 4;
    const auto kernel = layer_first_kernel<TOKENS, CAP, DECODED, C, U, LARGE>;
    static bool ready[64];                       // (per device; setting the attribute twice does no harm)
    int dev = 0;
    PM_REQUIRE(hipGetDevice(&dev) == hipSuccess, "%s: no device", who);
    if (dev >= 64 || !ready[dev]) {
        PM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess,
                   "%s: the kernel needs %d bytes of LDS", who, LDS);
        if (dev < 64) ready[dev] = true;
    }
    kernel<<<dim3((unsigned)((p.N + COLS - 1) / COLS), (unsigned)p.batches), FIRST_WAVES * 64, LDS, stream>>>(p, r);
    PM_LAUNCH_CHECK(who);
    return 0;
}

// Up to 32 tokens (one routing group), 16 experts, 4 choices and 16 rows an expert, and a compute unit for each work-group: a second
// round of work-groups would route once more.  (Rows are below 4 MB, as the products ask for, so that one descriptor covers x.)
static bool first_serves(int dtype, int fp32_gate, int samples, int model_dim, int experts, int top_k, int capacity, int hidden)
{
    if (dtype != PLANMOE_BF16 || !fp32_gate || samples > FIRST_TOKENS || experts > 16 || (top_k < experts ? top_k : experts) > 4) return false;
    if (capacity < 1 || capacity > FIRST_ROWS || (int64_t)hidden * model_dim * 2 >= ((int64_t)1 << 31)) return false;
    const int width = gemm_skinny_width(false, hidden, model_dim, experts);
    return (int64_t)((hidden + width - 1) / width) * experts <= compute_units();
}

} // namespace pm

using namespace pm;

extern "C" int planmoe_layer_dispatch_product(const void *x, const void *wg, int dtype, int fp32_gate, int samples, int model_dim,
                                              int experts, int top_k, int normalize_gate, int capacity, int codec,
                                              int32_t *indices, int32_t *locations, void *gates, int64_t plane_stride,
                                              float *l_aux, int32_t *expert_counts, const void *w1, const void *b1, int hidden,
                                              int rows_hint, void *rows, void *h, void *workspace, size_t workspace_bytes,
                                              void *stream)
{
    const char *who = "planmoe_layer_dispatch_product";
    PM_REQUIRE(expert_counts, "%s: NULL routing output", who);
    PM_REQUIRE(top_k >= 1, "%s: bad shape", who);
    // what the product would refuse, before anything is enqueued: its operands' ranges (the rows come from x where there is one launch), too
    if (expert_gemm_check(who, 0, dtype, x, w1, experts, capacity, hidden, model_dim, expert_counts, top_k < experts ? top_k : experts, 1, h)) return 1;
    const bool shape = wg && indices && locations && gates && samples >= 1 && plane_stride >= samples && (codec == 0 || codec == 1) && aligned16(wg);
    // (a call that is not well formed goes on to the entry point that says what is wrong with it)
    if (!shape || !first_serves(dtype, fp32_gate, samples, model_dim, experts, top_k, capacity, hidden)) {
        if (planmoe_layer_dispatch(x, wg, dtype, fp32_gate, nullptr, samples, model_dim, experts, top_k, normalize_gate, capacity, codec, indices, locations,
                                   gates, plane_stride, nullptr, l_aux, expert_counts, rows, workspace, workspace_bytes, stream)) return 1;
        return planmoe_expert_gemm(0, dtype, rows, w1, b1, 1, experts, capacity, hidden, model_dim, expert_counts, top_k < experts ? top_k : experts, 1,
                                   rows_hint, h, stream);
    }
    const SkinnyArgs p{nullptr, (const uint16_t *)w1, (const uint16_t *)b1, nullptr, (uint16_t *)h, nullptr, nullptr, 0, 1, capacity, hidden, model_dim, experts, 1};
    const FirstArgs r{x, wg, samples, top_k < experts ? top_k : experts, normalize_gate, indices, locations, gates, plane_stride, l_aux, expert_counts};
    hipStream_t st = (hipStream_t)stream;
    const int width = gemm_skinny_width(false, hidden, model_dim, experts);
    const bool large = skinny_large(hidden, model_dim, experts);
// (U8: steps on their way through the codec)
#define PM_FIRST__(TOKENS, C, U, U8, LARGE)                                                                              \
    (experts <= 8 ? (codec ? first_launch<TOKENS, 8, true, C, U8, LARGE>(p, r, st, who) : first_launch<TOKENS, 8, false, C, U, LARGE>(p, r, st, who))     \
                  : (codec ? first_launch<TOKENS, 16, true, C, U8, LARGE>(p, r, st, who) : first_launch<TOKENS, 16, false, C, U, LARGE>(p, r, st, who)))
#define PM_FIRST_(C, U, U8, LARGE) (samples <= 16 ? PM_FIRST__(16, C, U, U8, LARGE) : PM_FIRST__(FIRST_TOKENS, C, U, U8, LARGE))
#define PM_FIRST(C, U) (large ? PM_FIRST_(C, U, U, true) : PM_FIRST_(C, U, U, false))
    // (32 columns through the codec, whose values take registers: of eight steps seven registers were spilled, and a load that is spilled is waited
    // for.  us, 1 token, weights in the last cache and cold, two launches, eight steps, four:
    //   8 experts, 1024 -> 1024   11.7, 10.8, 9.1    13.0, 13.3, 10.6      4 experts, 4096 -> 2048   22.6, 31.7, 22.9    29.8, 33.8, 25.3
    //   8 experts, 2048 -> 1024   14.8, 17.7, 13.8   18.6, 20.1, 17.0      8 experts, 4096 -> 1024   21.4, 31.2, 22.7    29.3, 33.2, 25.4)
    // (and not nontemporally, see gemm_skinny.hip: without the codec, 1 token, nontemporal and not, 8 experts, 4096 -> 1024 22.2, 18.3 and 24.8, 25.5;
    // 4 experts, 4096 -> 2048 22.5, 17.9 and 24.3, 25.4; 8 experts, 8192 -> 1024 38.5, 28.7 and 40.7, 40.2)
    return width == 32 ? PM_FIRST_(2, 8, 4, false) : width == 64 ? PM_FIRST(4, 2) : PM_FIRST(8, 1);
#undef PM_FIRST
#undef PM_FIRST_
#undef PM_FIRST__
}
