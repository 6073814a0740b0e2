// The layer's second product and the combine behind it.
//
// Where the product has few columns the weight is read by few compute units, and one compute unit gets at most 28 GB/s from memory
// (8 experts of 32 rows, 4096 -> 1024: 128 tiles of 128 x 64, 31 us with the combine for 67 MB).  There its reduction is divided between work-groups that
// each leave fp32 sums in a plane of their own, and the combine, which reads the rows anyway, adds the planes of a row, rounds, adds the
// bias and rounds again, as the product's own epilogue would: no work-group waits for another and no launch is added (22.5 us).
// The shares are written and read once, beside 67 MB of weights: 256 rows of 1024 values 1 MB each.  Where that takes longer than it saves is
// gemm_shares_pay's rule.
#include "rows.hpp"
#include "int8_core.hpp"
#include "layer_rows.hpp"
#include "layer_shares.hpp"

namespace pm {

// without a codec: out[t] = sum_j gate_j * row(slot_j), planes left to right, one rounding at the end.  A wave has 512 columns of a token.
// rows_out: the rows of the tokens are kept.
template <bool KEEP>
__global__ __launch_bounds__(256) void combine_shares_kernel(const RowShares rows, const float *__restrict__ gates, const int32_t *__restrict__ indices,
                                                             const int32_t *__restrict__ locations, int64_t stride, int top_k, int samples, int chunks,
                                                             uint16_t *__restrict__ rows_out, uint16_t *__restrict__ out)
{
    using E = Elem<PLANMOE_BF16>;
    const int lane = lane_id(), id = blockIdx.x * 4 + (threadIdx.x >> 6), t = id / chunks, units = rows.model_dim / 8;
    if (t >= samples) return;
    const int u = id % chunks * WAVE + lane;
    int slot; float gate;
    fetch_planes(gates, indices, locations, stride, t, 0, top_k, 0x7fffffff, rows.capacity, slot, gate);
    float acc[8];
    for (int j = 0; j < top_k; ++j) {
        const int s = rl_i(slot, j);
        const float g = rl_f(gate, j);
        const uint4 row = rows.vector(max(s, 0), min(u, units - 1));
        if (KEEP && s >= 0 && u < units) stream_store(reinterpret_cast<uint4 *>(rows_out + (int64_t)s * rows.model_dim) + u, row);
        float f[8];
        E::unpack(row, f);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float v = s >= 0 ? g * f[i] : 0.f;
            acc[i] = j == 0 ? v : acc[i] + v;
        }
    }
    if (u < units) stream_store(reinterpret_cast<uint4 *>(out + (int64_t)t * rows.model_dim) + u, E::pack(acc));
}

// The planes have a row for every slot, used or not, so a capacity far beyond the rows that are expected (no token dropped: as many slots an expert
// as there are tokens) would have them take many times what is read: 64 experts of 8192 slots x 128 values, 4 shares, 1 GB beside rows of 134 MB.
// The rows in use of a chip full of tiles are 17 MB altogether; four times that is where shares become fewer, or the product whole.
constexpr int64_t SHARES_BYTES = (int64_t)64 << 20;

static int rows_expected(int rows_hint, int capacity) { return rows_hint >= 1 && rows_hint < capacity ? rows_hint : capacity; }

static GemmShares shares_of(int dtype, int codec, int hidden, int top_k, int samples, int model_dim, int experts, int capacity, int rows_hint)
{
    // (vectors of 8 values, up to 64 choices a lane each, rows of the codec's kernel in registers; elsewhere the general path)
    if (dtype != PLANMOE_BF16 || (codec != 0 && codec != 1) || hidden < 8 || hidden % 8 != 0 || model_dim < 8 || model_dim % 8 != 0 || model_dim > 4096) return GemmShares{};
    if (experts < 1 || experts > 64 || top_k < 1 || top_k > experts || samples < 1 || capacity < 1) return GemmShares{};
    if ((int64_t)(hidden > model_dim ? hidden : model_dim) * 512 >= ((int64_t)1 << 31) || (int64_t)experts * capacity >= ((int64_t)1 << 31)) return GemmShares{};
    const int64_t most = SHARES_BYTES / ((int64_t)experts * capacity * model_dim * 4);
    return gemm_shares_pick(capacity, model_dim, hidden, experts, rows_expected(rows_hint, capacity), (int64_t)samples * top_k, most);
}

} // namespace pm

using namespace pm;

extern "C" int planmoe_layer_product_combine_pays(int dtype, int codec, int hidden, int top_k, int samples, int model_dim, int experts, int capacity, int rows_hint)
{
    const GemmShares how = shares_of(dtype, codec, hidden, top_k, samples, model_dim, experts, capacity, rows_hint);
    return how.splits > 0 && gemm_shares_pay(how, capacity, model_dim, hidden, experts, rows_expected(rows_hint, capacity), (int64_t)samples * top_k, codec == 1);
}

extern "C" size_t planmoe_layer_product_combine_workspace_bytes(int dtype, int codec, int hidden, int top_k, int samples, int model_dim,
                                                                int experts, int capacity, int rows_hint)
{
    const GemmShares how = shares_of(dtype, codec, hidden, top_k, samples, model_dim, experts, capacity, rows_hint);
    return (size_t)how.splits * experts * capacity * model_dim * 4;
}

extern "C" int planmoe_layer_product_combine(const void *h, const void *w2, const void *b2, int dtype, int codec, int hidden, const float *gates,
                                             const int32_t *indices, const int32_t *locations, int64_t plane_stride, int top_k,
                                             int samples, int model_dim, int experts, int capacity, const int32_t *expert_counts,
                                             int count_round, int rows_hint, void *rows, int keep_rows, uint8_t *codes, void *bias,
                                             void *scale, void *out, void *workspace, size_t workspace_bytes, void *stream)
{
    const char *who = "planmoe_layer_product_combine";
    if (layer_rows_check(who, dtype, rows, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, codec)) return 1;
    PM_REQUIRE(expert_counts && count_round >= 1, "%s: NULL counts, or they are rounded up to multiples of less than 1", who);
    PM_REQUIRE(!codes || (codec == 1 && bias && scale && aligned16(codes)), "%s: codes are kept with their minima and scales, 16-byte aligned, of the int8 codec", who);
    if (samples == 0) return 0;
    PM_REQUIRE(out && aligned16(out), "%s: NULL or unaligned output", who);
    const GemmShares how = count_round == 1 ? shares_of(dtype, codec, hidden, top_k, samples, model_dim, experts, capacity, rows_hint) : GemmShares{};
    if (how.splits == 0) {
        if (planmoe_expert_gemm(0, dtype, h, w2, b2, 0, experts, capacity, model_dim, hidden, expert_counts, top_k, count_round, rows_hint, rows, stream)) return 1;
        if (codes) return planmoe_layer_combine_keep(rows, dtype, gates, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, out, codes, bias, scale, stream);
        return planmoe_layer_combine(rows, dtype, codec, gates, indices, locations, plane_stride, top_k, samples, model_dim, experts, capacity, out, stream);
    }
    PM_REQUIRE(h && w2 && aligned16(h) && aligned16(w2), "%s: NULL or unaligned operand", who);
    PM_REQUIRE(!b2 || (uintptr_t)b2 % 2 == 0, "%s: unaligned bias", who);
    PM_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= planmoe_layer_product_combine_workspace_bytes(dtype, codec, hidden, top_k, samples,
               model_dim, experts, capacity, rows_hint), "%s: workspace too small", who);
    hipStream_t st = (hipStream_t)stream;
    SkinnyArgs p{(const uint16_t *)h, (const uint16_t *)w2, nullptr, nullptr, nullptr, nullptr, expert_counts, top_k, 1, capacity, model_dim, hidden, experts, 0};
    p.shares = (float *)workspace;
    if (gemm_shares_run(how, p, st, who)) return 1;
    const RowShares shares{(const float *)workspace, (int64_t)experts * capacity * model_dim, how.splits, (const uint16_t *)b2, capacity, model_dim};
    if (codec) return combine_int8_shares(who, shares, gates, indices, locations, plane_stride, top_k, samples, out, codes, bias, scale, st);
    const int chunks = (model_dim / 8 + WAVE - 1) / WAVE;
    const unsigned blocks = (unsigned)(((int64_t)samples * chunks + 3) / 4);
    if (keep_rows) combine_shares_kernel<true><<<blocks, 256, 0, st>>>(shares, gates, indices, locations, plane_stride, top_k, samples, chunks, (uint16_t *)rows, (uint16_t *)out);
    else combine_shares_kernel<false><<<blocks, 256, 0, st>>>(shares, gates, indices, locations, plane_stride, top_k, samples, chunks, nullptr, (uint16_t *)out);
    PM_LAUNCH_CHECK(who);
    return 0;
}
