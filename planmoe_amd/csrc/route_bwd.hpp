// The routing's backward pass of one token, by a group of lanes (as many as there are experts, a power of two, at most a wave): how
// the scores' gradient follows from the gates' and the GShard loss's.
//   g_j = s_j / D, D = max(sum_i s_i, eps)  =>  ds_j = (dg_j - [sum >= eps] * sum_i dg_i g_i) / D
//   l_aux = sum_e me[e] ce[e] / T            =>  ds[t][e] += dl * ce[e] / T,  ce[e] = count0[e] * E / T
//   softmax: dlogit_e = s_e * (ds_e - sum_i ds_i s_i)
#pragma once
#include "common.hpp"

namespace pm {

struct RouteBwd {
    const void *scores;                          // [samples, experts]
    const float *dl_aux;                         // NULL: the loss has no gradient
    const int *count0;
    int samples, experts, k, normalize, group;
};
inline int route_bwd_group(int experts)
{
    int group = 1;
    while (group < experts && group < WAVE) group <<= 1;
    return group;
}

// expert(j), dgate(j): the token's choice j and its gate's gradient in the scores' precision; e0: the lane's place in its group, all of
// which are here.  put(e, v): the gradient of the token's score e, or of its logit.
template <int DT, typename Expert, typename Dgate, typename Put>
__device__ __forceinline__ void route_bwd_token(const RouteBwd &r, int t, int e0, bool through_softmax, Expert expert, Dgate dgate, Put put)
{
    using E = Elem<DT>;
    const int64_t base = (int64_t)t * r.experts;
    const float dl = r.dl_aux ? r.dl_aux[0] : 0.f;
    const float lscale = dl * ((float)r.experts / (float)r.samples) / (float)r.samples;
    float sum = 0.f, dot = 0.f;
    for (int j = 0; j < r.k; ++j) {
        const int e = expert(j);
        if (e < 0 || e >= r.experts) continue;           // (no expert: the choice is not there)
        const float sj = E::load(r.scores, base + e);
        sum = E::round(sum + sj);
        dot += dgate(j) * sj;
    }
    const float eps = DT == PLANMOE_F32 ? 1.1920928955078125e-07f : DT == PLANMOE_BF16 ? 0.0078125f : 0.0009765625f;
    const bool norm = r.k > 1 && r.normalize;
    const float D = norm ? fmaxf(sum, eps) : 1.f;
    const float corr = (norm && sum >= eps) ? dot / (D * D) : 0.f;      // sum_i dg_i g_i / D
    auto ds_at = [&](int e) {
        float v = r.count0 ? lscale * (float)r.count0[e] : 0.f;
        for (int j = 0; j < r.k; ++j)
            if (expert(j) == e) v += dgate(j) / D - corr;
        return v;
    };
    if (!through_softmax) {
        for (int e = e0; e < r.experts; e += r.group) put(e, ds_at(e));
    } else {
        float inner = 0.f;
        for (int e = e0; e < r.experts; e += r.group) inner += ds_at(e) * E::load(r.scores, base + e);
        for (int d = 1; d < r.group; d <<= 1) inner += __shfl_xor(inner, d);
        for (int e = e0; e < r.experts; e += r.group) {
            const float s = E::load(r.scores, base + e);
            put(e, s * (ds_at(e) - inner));
        }
    }
}

} // namespace pm
