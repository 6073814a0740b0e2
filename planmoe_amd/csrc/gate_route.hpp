// A routing group as one work-group of four waves has it: the gate's logits, softmax, choices, gates and ranks.  What gate_route_kernel
// (forward.hip) is made of, and what the layer's first product for few tokens starts with (layer_first.hip).
#pragma once
#include "forward_shared.hpp"

namespace pm {

// tokens per work-group of the gate kernel = tokens per routing group (one lane each in the
// routing epilogue): 64, or fewer where 64 would leave compute units without a work-group; row_bytes: of a token
inline int fwd_group_tokens(int experts, int samples, int64_t row_bytes)
{
    const int cu = compute_units();
    // measured at 8 experts: 16384 tokens (256 groups of 64) 39 us with 64, 44 us with 32;
    // 8192 tokens 32 us with 64, 28 us with 32.  One compute unit gets some 30 GB/s, so fewer tokens in a group are fewer bytes in that chain, up to one
    // group a compute unit; beyond, two groups on some units take longer than one of 32.  us of the send side with 32 and with 16 tokens:
    //   bf16, 8 x 2048    40 tokens 13.3, 11.5   1999 16.9, 14.9   4096 20.5, 19.0   5000 20.1, 22.0
    //   bf16, 16 x 512    40 tokens 11.9, 10.9   1999 14.2, 13.1   4096 17.0, 14.5
    //   bf16, 16 x 4096   40 tokens 22.1, 17.3   1999 25.1, 20.4   4096 34.1, 28.2   5000 36.4, 38.0
    //   fp32, 16 x 1024   40 tokens 15.9, 13.1   1999 19.7, 16.7   4096 24.1, 19.6   5000 23.4, 24.6
    //   fp32, 8 x 4096    40 tokens 32.5, 25.9   1999 38.8, 31.7   4096 50.9, 48.4   5000 56.2, 64.1
    // With up to 8 experts from rows of 2 KB on: below, the bytes are few, and more groups are more columns to sum behind them.
    //   bf16, 8 x 256     40 tokens 9.4, 9.5     200  9.6, 9.8     4096 12.8, 13.0
    //   bf16, 8 x 512     40 tokens 9.5, 9.8     200 10.0, 10.5    4096 14.0, 14.1      8 x 1024   10.9, 10.7   11.4, 11.2   16.4, 16.1
    //   fp32, 8 x 256     40 tokens 9.1, 9.4     200  9.9, 10.5    4096 14.0, 14.2      8 x 512    10.8, 10.8   11.0, 11.1   16.4, 16.6
    //   fp32, 4 x 512     40 tokens 9.0, 9.0     200  9.5, 9.3     4096 13.4, 13.4      8 x 768    11.8, 10.9   12.4, 11.5   18.9, 18.1
    // Up to 32 tokens are one group, and one launch (plan.one); up to 16 of them have the products of 16, half the loads and in fp32 half the matrix cores' time.  us of a layer's pass on the GPU with 32 and with 16,
    // 8 tokens: bf16, 8 x 1024 -> 4096 37.5, 36.0; 16 x 3840 -> 256 35.3, 32.8
    if (experts <= 16) {
        if (samples <= 16) return 16;
        return samples > 32 && samples <= 16 * cu && (experts > 8 || row_bytes >= 2048) ? 16 : samples < 64 * cu ? 32 : 64;
    }
    // as many groups as compute units at most (16 tokens: where four waves find a share of the experts).  us of the send side, bf16, with 64, 32, 16:
    //   64 experts x 1368   48 tokens 26, 22, 21;  4074 33, 29, 27;  8000 35, 32, 42;  16000 39, 47, 74
    //   32 experts x 1368   48 tokens 24, 20;      4074 33, 24;      8000 35, 28;      16000 42, 42
    if (experts > 32 && samples <= 16 * cu) return 16;
    return samples <= 32 * cu ? 32 : 64;
}
constexpr int FWD_LOSS_PARTS = 64;
inline void *fwd_tables(void *workspace) { return (char *)workspace + FWD_TABLES_OFFSET; }

// hist_t / me_t are the transposes of hist / me with the group index running fastest (rows of
// gstride = groups rounded up to 4 entries, the padding zero): a column of the histogram, which
// is what a prefix over groups reads, is contiguous there.
struct FwdWs {
    int32_t *totals, *hist, *offs, *rank, *hist_t;
    float *loss_part, *me, *row_min, *row_max, *me_t;
    int gstride;
};
__host__ __device__ inline size_t fwd_pad4(size_t words) { return (words + 3) & ~(size_t)3; }
__host__ __device__ inline FwdWs fwd_ws(void *ws, int groups, int k, int experts, int samples)
{
    FwdWs w;
    w.gstride = (int)fwd_pad4((size_t)groups);
    w.hist_t = (int32_t *)ws;                                   // 16-byte aligned rows
    w.me_t = (float *)(w.hist_t + (size_t)k * experts * w.gstride);
    w.totals = (int32_t *)(w.me_t + (size_t)experts * w.gstride);
    w.loss_part = (float *)(w.totals + experts);
    w.hist = (int32_t *)(w.loss_part + FWD_LOSS_PARTS);
    w.offs = w.hist + (size_t)groups * k * experts;
    w.me = (float *)(w.offs + (size_t)groups * k * experts);
    w.rank = (int32_t *)(w.me + (size_t)groups * experts);
    w.row_min = (float *)(w.rank + (size_t)k * samples);
    w.row_max = w.row_min + samples;
    return w;
}

// OUT: what a kept row arrives as.  CODES: codes with bias and scale.  ROWS: no codec -- `codes` is the
// dispatched buffer in x's dtype and a kept row arrives there as 0 + x (what fast_encode's accumulation
// into zeros leaves: -0 becomes +0), an empty slot as zeros.  DECODED: the same buffer with what the
// decompressor makes of the row's codes (the codes stay in registers: one pass where dispatch + int8
// and the decompressor write and read them).
enum { OUT_CODES = 0, OUT_ROWS = 1, OUT_DECODED = 2 };
// SDT: dtype of logits / scores / gates (F32 when fp32_gate, else the input dtype)
// CAP: compile-time bound of the expert count held in registers by the routing epilogue
// NT == 1: split-K over the 4 waves, weights straight from L2 (up to 16 experts);
// NT > 1: weights shared through LDS, a wave per 16 tokens.
// MODE 0: logits = x . wg^T computed here.  MODE 1 / 2: no GEMM; x holds the [samples, experts]
// logits / scores in the routing dtype (the stand-alone routing entry point) and only the
// epilogue runs.
// ONE (not ONE_OFF): all tokens are one group, so what the group knows is all there is, and slots, loss and counts are
// final.  OUT_ROWS / OUT_DECODED: the rows go to their slots as well; every work-group routes all tokens for itself, sends the
// rows of four, and the first one writes the routing.  (A pass of the layer at 8 tokens x 1024, hidden 4096, 8 experts: 51.0 us
// with two launches for this, 47.1 with one; the copy itself is 16 KB.)
enum { ONE_OFF = -1, ONE_ROUTING = 0 };

template <int DT, int NT, int CAP, bool SPLITK, int GROUP, int MODE, int ONE>
struct GateShared {
    static constexpr int COLS = 16 * NT + 1;
    static constexpr bool STATS = DT == PLANMOE_BF16 && MODE == 0;
    // split-K: part[4][GROUP][COLS] floats; else the weight buffers / logits[GROUP][COLS]
    uint4 smem[SPLITK ? (4 * GROUP * COLS + 3) / 4 : gate_lds_vectors<NT>()];
    int32_t hist[CAP];
    int32_t pstat[STATS && SPLITK ? 4 : 1][STATS ? GROUP : 1][3];
    uint8_t best[64][GROUP];                           // [plane][token] chosen expert
    float me[4][CAP];
    int32_t slot[ONE > 0 ? 4 : 1][GROUP];              // (ONE) a choice's slot, -1: none
    int32_t total[ONE > 0 ? CAP : 1];                  // (ONE) choices of an expert
    float range[ONE == OUT_DECODED && STATS ? GROUP : 1][2];
};

// Group `block` of `groups`; with ONE, where several work-groups route the same tokens, the `first` writes the routing.
// Two barriers; what is left in `sh` is there behind another.
// DEPTH: steps of the products on their way, up to 16 experts
template <int DT, int SDT, int NT, int CAP, bool SPLITK, int GROUP, int MODE, int ONE, int DEPTH = GROUP == 16 ? 4 : 2>
__device__ __forceinline__ void gate_route_group(
    GateShared<DT, NT, CAP, SPLITK, GROUP, MODE, ONE> &sh, bool first, int block, int groups,
    const void *__restrict__ x, const void *__restrict__ wg, const float *__restrict__ logit_bias,
    int samples, int model_dim, int experts, int k, int normalize_gate,
    int32_t *__restrict__ indices, int32_t *__restrict__ locations, void *__restrict__ gates,
    int64_t stride, void *__restrict__ logits_out, void *__restrict__ scores_out,
    float *__restrict__ l_aux, int32_t *__restrict__ counts_out, void *__restrict__ workspace, int capacity)
{
    using S = Elem<SDT>;
    static_assert(GROUP == 64 || GROUP == 32 || GROUP == 16, "tokens of a group");
    constexpr int COLS = 16 * NT + 1;
    auto &smem = sh.smem;
    auto &s_hist = sh.hist;
    float (*part)[GROUP][COLS] = reinterpret_cast<float (*)[GROUP][COLS]>(smem);

    const int tid = threadIdx.x, lane = lane_id();
    const FwdWs ws = fwd_ws(workspace, groups, k, experts, samples);
    const int t0 = ONE == ONE_OFF ? block * GROUP : 0;
    // the additive logit biases of this lane's experts, asked for before the GEMM: read where they are
    // used, their latency would stand in every pass of the epilogue (6.5 -> 2 us per group at 64 experts)
    constexpr int LPT_ = CAP < 16 ? CAP : 16, EPL_ = CAP / LPT_;
    float lbias[EPL_];
#pragma unroll
    for (int q = 0; q < EPL_; ++q) {
        const int e = q * LPT_ + lane % LPT_;
        lbias[q] = (MODE != 2 && logit_bias && e < experts) ? logit_bias[e] : 0.f;
    }
    constexpr bool STATS = DT == PLANMOE_BF16 && MODE == 0;
    static_assert(MODE == 0 || !SPLITK, "routing from memory has one part");
    auto &pstat = sh.pstat;
    if constexpr (MODE != 0) {
        // the group's rows land where the GEMM would have left its logits: 8 loads in flight per
        // thread, at clamped indices so that they are straight-line loads
        const int n = min(GROUP, samples - t0) * experts;
        const int64_t base = (int64_t)t0 * experts;
        for (int i0 = tid; i0 < n; i0 += 8 * 256) {
            float v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = S::load(x, base + min(i0 + q * 256, n - 1));
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int i = i0 + q * 256;
                if (i < n) {
                    const int tok = i / experts;
                    part[0][tok][i - tok * experts] = v[q];
                }
            }
        }
    } else if constexpr (SPLITK) {
        // (DEPTH: groups of 32, two on some compute units: 8 x 4096 fp32, 6500 tokens 68 us with two, 70 with four)
        if constexpr (STATS) gate_tile_partials<DT, NT, GROUP / 16, 4, true, DEPTH>(x, wg, t0, samples, model_dim, experts, part, pstat);
        else gate_tile_partials<DT, NT, GROUP / 16, 4, false, DEPTH>(x, wg, t0, samples, model_dim, experts, part);
    } else {
        if constexpr (STATS) gate_tile_lds<DT, NT, true, GROUP>(x, wg, t0, samples, model_dim, experts, smem, pstat[0]);
        else gate_tile_lds<DT, NT, false, GROUP>(x, wg, t0, samples, model_dim, experts, smem);
    }
    __syncthreads();

    // ---- routing epilogue, part 1: all four waves, wave w owns GROUP / 4 consecutive tokens.
    // LPT lanes share a token, lane el holding the experts el, el + LPT, ...: softmax and the
    // k-fold arg-max are butterflies over those lanes instead of loops over the experts.
    constexpr int LPT = CAP < 16 ? CAP : 16;           // lanes per token
    constexpr int EPL = CAP / LPT;                     // experts per lane
    constexpr int TPW4 = GROUP / 4;                    // tokens per wave
    constexpr int TPP = WAVE / LPT < TPW4 ? WAVE / LPT : TPW4;   // tokens per pass of a wave
    auto &s_best = sh.best;
    auto &s_me = sh.me;
    const int wave = tid >> 6, el = lane % LPT, tk = lane / LPT;
    auto token_reduce = [&](auto v, auto op) { return row_allreduce<LPT>(v, op); };   // over the lanes of a token
    float me_acc[EPL];
#pragma unroll
    for (int q = 0; q < EPL; ++q) me_acc[q] = 0.f;
    const float eps = SDT == PLANMOE_F32 ? 1.1920928955078125e-07f
                    : SDT == PLANMOE_BF16 ? 0.0078125f : 0.0009765625f;

    for (int p = 0; p < TPW4 / TPP; ++p) {
        const int tok = wave * TPW4 + p * TPP + min(tk, TPP - 1);   // lanes past the pass repeat a token
        const int t = t0 + tok;
        const bool valid = t < samples && tk < TPP, writes = valid && first;
        float sc[EPL];
        float mx = -INFINITY;
        bool lost = false;                                // (MODE 0, 1) the token's scores are NaN
#pragma unroll
        for (int q = 0; q < EPL; ++q) {
            const int e = q * LPT + el;
            float v = -INFINITY;
            if (e < experts) {
                if constexpr (SPLITK) v = ((part[0][tok][e] + part[1][tok][e]) + part[2][tok][e]) + part[3][tok][e];
                else v = part[0][tok][e];
                v = S::round(v);
                if constexpr (MODE != 2) {
                    if (logits_out && writes) S::store(logits_out, (int64_t)t * experts + e, v);
                    if (logit_bias) v = S::round(v + lbias[q]);
                }
            }
            sc[q] = v;                                    // MODE 2: the score itself (-inf past the experts)
            mx = fmaxf(mx, v);
        }
        if constexpr (MODE != 2) {
            mx = token_reduce(mx, [](float a, float b) { return fmaxf(a, b); });
            float sum = 0.f;
#pragma unroll
            for (int q = 0; q < EPL; ++q) {
                sc[q] = (q * LPT + el < experts) ? expf(sc[q] - mx) : 0.f;
                sum += sc[q];
            }
            sum = token_reduce(sum, [](float a, float b) { return a + b; });
            const float inv = 1.0f / sum;                 // scores are tolerance-level quantities
            lost = sum != sum;
#pragma unroll
            for (int q = 0; q < EPL; ++q) {
                const int e = q * LPT + el;
                if (e < experts) {
                    sc[q] = S::round(sc[q] * inv);
                    if (scores_out && writes) S::store(scores_out, (int64_t)t * experts + e, sc[q]);
                } else {
                    sc[q] = -INFINITY;
                }
            }
        }
        // column sums of the wave's scores (GShard loss): over the tokens of the pass, then passes
        if (l_aux) {
#pragma unroll
            for (int q = 0; q < EPL; ++q) {
                float c = (valid && q * LPT + el < experts) ? sc[q] : 0.f;
#pragma unroll
                for (int off = LPT; off < WAVE; off <<= 1) c += __shfl_xor(c, off, WAVE);   // lanes past the pass hold 0
                me_acc[q] += c;
            }
        }
        // k-fold arg-max, the lower expert id wins among equal scores.  Behind the softmax a token's scores are all NaN or none is: then they
        // are all the same (NaN compared as such, as scores that came from outside are, costs 1.2 us in 65 at 32768 tokens x 64 experts)
        if constexpr (MODE != 2) {
#pragma unroll
            for (int q = 0; q < EPL; ++q) sc[q] = lost ? 0.f : sc[q];
        }
        auto above = [](float a, float b) { if constexpr (MODE == 2) return score_above(a, b); else return a > b; };
        auto same = [](float a, float b) { if constexpr (MODE == 2) return score_same(a, b); else return a == b; };
        uint32_t taken = 0;
        float denom = 0.f, my_gate = 0.f;
        int my_idx = 0;
        for (int j = 0; j < k; ++j) {
            float bv = -INFINITY; int bi = 0x7fffffff;
#pragma unroll
            for (int q = 0; q < EPL; ++q) {
                const bool free_ = !((taken >> q) & 1u) && q * LPT + el < experts;
                if (free_ && (bi == 0x7fffffff || above(sc[q], bv))) { bv = sc[q]; bi = q * LPT + el; }
            }
            auto merge = [&](float ov, int oi) {
                const bool better = oi != 0x7fffffff && (bi == 0x7fffffff || above(ov, bv) || (oi < bi && same(ov, bv)));
                if (better) { bv = ov; bi = oi; }
            };
            if constexpr (LPT >= 2) merge(row_partner<1>(bv), row_partner<1>(bi));
            if constexpr (LPT >= 4) merge(row_partner<2>(bv), row_partner<2>(bi));
            if constexpr (LPT >= 8) merge(row_partner<4>(bv), row_partner<4>(bi));
            if constexpr (LPT >= 16) merge(row_partner<8>(bv), row_partner<8>(bi));
#pragma unroll
            for (int q = 0; q < EPL; ++q) if (bi == q * LPT + el) taken |= 1u << q;
            if (MODE != 2 && lost) bv = NAN;
            denom = (j == 0) ? bv : S::round(denom + bv);
            if (el == 0 && tk < TPP) s_best[j][tok] = (uint8_t)bi;
            if (j < LPT) {
                if (el == j) { my_gate = bv; my_idx = bi; }
            } else if (writes && el == j % LPT) {
                // more planes than lanes per token: index and raw gate go out now, the gate is
                // normalised below
                indices[(int64_t)j * stride + t] = bi;
                S::store(gates, (int64_t)j * stride + t, bv);
            }
        }
        if (writes) {
            const bool norm = k > 1 && normalize_gate;
            const float d = fmaxf(denom, eps);
            if (el < k) {
                indices[(int64_t)el * stride + t] = my_idx;
                S::store(gates, (int64_t)el * stride + t, norm ? my_gate / d : my_gate);
            }
            if (norm) {
                for (int j = LPT + el; j < k; j += LPT) {
                    const float g = S::load(gates, (int64_t)j * stride + t);
                    S::store(gates, (int64_t)j * stride + t, g / d);
                }
            }
        }
    }
    if (l_aux && tk == 0) {
#pragma unroll
        for (int q = 0; q < EPL; ++q) if (q * LPT + el < experts) s_me[wave][q * LPT + el] = me_acc[q];
    }
    __syncthreads();

    auto &s_slot = sh.slot;
    auto &s_range = sh.range;
    // ---- part 2: wave 0, one lane per token: rank of every token among the group's tokens with
    // the same choice (wave ballots), the group's histograms, row min / max, score column sums
    if (tid < WAVE) {
        const int t = t0 + tid;
        const bool valid = tid < GROUP && t < samples;
        if constexpr (STATS) {
            if (valid) {
                // row min / max for the int8 codec of the dispatch launch
                int a = pstat[0][tid][0], b = pstat[0][tid][1], n = pstat[0][tid][2];
                if constexpr (SPLITK) {
#pragma unroll
                    for (int w = 1; w < 4; ++w) {
                        a = min(a, pstat[w][tid][0]); b = max(b, pstat[w][tid][1]); n = max(n, pstat[w][tid][2]);
                    }
                }
                float lo, hi;
                RowStats<PLANMOE_BF16, true>::decode(a, b, n, lo, hi);
                if constexpr (ONE == ONE_OFF) { ws.row_min[t] = lo; ws.row_max[t] = hi; }
                else if constexpr (ONE == OUT_DECODED) { s_range[tid][0] = lo; s_range[tid][1] = hi; }
            }
        }
        if (l_aux && lane < experts) {
            const float v = ((s_me[0][lane] + s_me[1][lane]) + s_me[2][lane]) + s_me[3][lane];
            if constexpr (ONE == ONE_OFF) {
                ws.me[(int64_t)block * experts + lane] = v;
                ws.me_t[(int64_t)lane * ws.gstride + block] = v;
            } else {
                s_me[0][lane] = v;
            }
        }
        int before = 0;                                            // ONE: entries of expert `lane` in the planes before
        for (int j = 0; j < k; ++j) {
            const int best = valid ? (int)s_best[j][tid % GROUP] : -1;
            if (lane < CAP) s_hist[lane] = 0;
            __builtin_amdgcn_wave_barrier();
            int rank = 0;
            if constexpr (CAP <= 16) {
                // few experts: one ballot per expert, no serial dependence between them
#pragma unroll
                for (int e = 0; e < CAP; ++e) {
                    const uint64_t m = __ballot(best == e);
                    if (best == e) rank = __popcll(m & lanes_below());
                    if (lane == e) s_hist[e] = __popcll(m);
                }
            } else {
                uint64_t todo = __ballot(valid);
                while (todo) {
                    const int leader = __ffsll((unsigned long long)todo) - 1;
                    const int le = __builtin_amdgcn_readlane(best, leader);
                    const uint64_t m = __ballot(valid && best == le);
                    if (valid && best == le) rank = __popcll(m & lanes_below());
                    if (lane == leader) s_hist[le] = __popcll(m);
                    todo &= ~m;
                }
            }
            if (ONE == ONE_OFF && valid) ws.rank[(int64_t)j * samples + t] = rank;
            __builtin_amdgcn_wave_barrier();
            if constexpr (ONE != ONE_OFF) {
                const int l = rank + __shfl(before, max(best, 0));
                if (valid && first) locations[(int64_t)j * stride + t] = l;
                if constexpr (ONE > 0) { if (tid < GROUP) s_slot[j][tid] = valid && l < capacity ? best * capacity + l : -1; }
                const int n = lane < experts ? s_hist[lane] : 0;
                before += n;
                if (lane < experts && first) {
                    if (counts_out) counts_out[j * experts + lane] = n;
                    if (j == 0 && l_aux) s_me[1][lane] = s_me[0][lane] * ((float)n * ((float)experts / (float)samples));
                }
            } else if (lane < experts) {
                ws.hist[((int64_t)block * k + j) * experts + lane] = s_hist[lane];
                int32_t *col = ws.hist_t + ((int64_t)j * experts + lane) * ws.gstride;
                col[block] = s_hist[lane];
                if (block == groups - 1)             // the last group also clears the padding
                    for (int p = groups; p < ws.gstride; ++p) col[p] = 0;
            }
            __builtin_amdgcn_wave_barrier();
        }
        if (ONE > 0 && lane < CAP) sh.total[lane] = before;
        if (ONE != ONE_OFF && l_aux && first && lane == 0) {
            float a = 0.f;
            for (int e = 0; e < experts; ++e) a += s_me[1][e];
            *l_aux = a / (float)samples;
        }
    }
}

} // namespace pm
