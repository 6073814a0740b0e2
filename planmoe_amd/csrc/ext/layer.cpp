// The layer with its built-in experts as one node: gate, routing, encode, codec, FFN, codec, decode, and
// the backward pass of all of them, driven from C++.
//
// A forward pass is four to nine launches of a few microseconds each at decode sizes; driven step by step
// from Python (an autograd node, a dozen tensor operations and a ctypes call with two dozen arguments for
// each) the host took 160 us for 40 us of GPU work.  Here a pass is one call: outputs and workspaces from
// torch's caching allocator, launches through the C ABI of libplanmoe_hip.
//
// With one rank the exchange delivers what was sent, so the "int8" codec is applied to rows in registers
// (planmoe_layer_dispatch, planmoe_layer_combine, planmoe_layer_combine_bwd) and the rows of empty capacity
// slots are neither written nor multiplied: the products get the number of rows in use of every expert.
#include "host.hpp"

namespace {

using namespace planmoe_host;

enum Codec { CODEC_NONE = 0, CODEC_INT8 = 1, CODEC_ZFP = 2, CODEC_LZ = 3 };
constexpr double ZFP_RATE = 8.0;             // zfpc.h:17

struct Shape {
    int T, M, E, H, k, cap, dt;
    int64_t rows() const { return (int64_t)E * cap; }
    // rows an expert is expected to have in use: what the products pick their tiles by
    int hint() const { return (int)std::min<int64_t>(cap, ((int64_t)T * k + E - 1) / E); }
    // what the second product leaves for the combine to add up, where that is the faster way
    size_t shares(int codec) const
    {
        if (codec > CODEC_INT8 || !planmoe_layer_product_combine_pays(dt, codec == CODEC_INT8, H, k, T, M, E, cap, hint())) return 0;
        return planmoe_layer_product_combine_workspace_bytes(dt, codec == CODEC_INT8, H, k, T, M, E, cap, hint());
    }
};

// which rows of an expert's buffer count: the tokens' own, a zfp block's four rows together, or (lz: the codec
// runs over the whole buffer) all of them
struct Live {
    const int32_t *counts;
    int planes, round;
};

// What the routing says, in one buffer that a backward pass keeps (a view or an allocation takes the host 1.5 - 2 us, and a training step of few
// tokens is the host's): indices [k, T], locations [k, T], counts [k, E], gates [k, T], scores [T, E]
struct Routing {
    Routing() = default;
    Routing(const Shape &s, at::ScalarType score_type) : type(score_type)
    {
        const int64_t each = score_type == at::kFloat ? 4 : 2, plane = (int64_t)s.k * s.T;
        auto piece = [&](int64_t n) { const int64_t at = words; words += (n + 255) / 256 * 64; return at; };
        idx_at = piece(plane * 4);
        loc_at = piece(plane * 4);
        cnt_at = piece((int64_t)s.k * s.E * 4);
        gates_at = piece(plane * each);
        scores_at = piece((int64_t)s.T * s.E * each);
    }
    void lie_in(const Tensor &buffer)
    {
        held = buffer;
        int32_t *base = buffer.data_ptr<int32_t>();
        idx = base + idx_at;
        loc = base + loc_at;
        cnt = base + cnt_at;
        gates = base + gates_at;
        scores = base + scores_at;
    }
    // the gates in fp32; `wide` holds what was converted
    const float *float_gates(const Shape &s, Tensor &wide) const
    {
        if (type == at::kFloat) return (const float *)gates;
        wide = at::from_blob(gates, {s.k, s.T}, held.options().dtype(type)).to(at::kFloat);
        return floats(wide);
    }
    at::ScalarType type = at::kFloat;
    int64_t words = 0, idx_at = 0, loc_at = 0, cnt_at = 0, gates_at = 0, scores_at = 0;
    Tensor held;
    int32_t *idx = nullptr, *loc = nullptr, *cnt = nullptr;
    void *gates = nullptr, *scores = nullptr;
};

struct Pass {
    Tensor y, l_aux, xe, h, ye, stream, codes;
    Routing r;
};

Tensor lz_round_trip(const Tensor &buf, void *st)
{
    const int64_t n = (int64_t)buf.nbytes(), blocks = planmoe_lz_blocks(n);
    Tensor offsets = at::empty({2, blocks + 1 + (-(blocks + 1) & 3)}, buf.options().dtype(at::kInt));      // (rows 16-byte aligned)
    Tensor flags = bytes(blocks * 64, buf), data = bytes(blocks * 2048, buf), ws = bytes((int64_t)planmoe_lz_workspace_bytes(n), buf);
    int32_t *fo = offsets.data_ptr<int32_t>(), *dof = fo + offsets.size(1);
    Tensor out = at::empty_like(buf);
    PM_CALL(planmoe_lz_compress(buf.data_ptr(), n, fo, dof, flags.data_ptr<uint8_t>(), data.data_ptr<uint8_t>(), ws.data_ptr(), (size_t)ws.numel(), st));
    PM_CALL(planmoe_lz_decompress(out.data_ptr(), n, fo, dof, flags.data_ptr<uint8_t>(), data.data_ptr<uint8_t>(), st));
    return out;
}

Tensor zfp_stream(const Shape &s, const Tensor &like) { return bytes((int64_t)planmoe_zfp_stream_bytes(2, s.M, s.rows(), ZFP_RATE), like); }

void zfp_rows(void *rows, const Tensor &stream, const Pass &p, const Shape &s, void *st)
{
    PM_CALL(planmoe_layer_zfp_rows((float *)rows, s.M, s.E, s.cap, p.r.cnt, s.k, raw(stream), stream.defined() ? (size_t)stream.numel() : 0, st));
}

Tensor zfp_workspace(const Shape &s, const Tensor &like) { return bytes((int64_t)planmoe_layer_zfp_workspace_bytes(s.E, s.cap), like); }

Live live_rows(const Pass &p, const Shape &s, int codec)
{
    if (codec == CODEC_LZ) return Live{nullptr, 1, 1};
    return Live{p.r.cnt, s.k, codec == CODEC_ZFP ? 4 : 1};
}

// a gradient as the kernels read rows: contiguous and 16-byte aligned (what comes back through torch.cat is contiguous,
// but begins anywhere)
Tensor as_rows(const Tensor &grad)
{
    const Tensor t = grad.contiguous();
    return (uintptr_t)t.data_ptr() % 16 == 0 ? t : t.clone(at::MemoryFormat::Contiguous);
}

// the codes of the experts' rows [rows, M], behind them the rows' minima and scales in x's dtype
struct Kept {
    Kept() = default;
    Kept(const Tensor &buffer, const Shape &s, int64_t size)
        : codes(buffer.data_ptr<uint8_t>()), bias(codes + s.rows() * s.M), scale(codes + s.rows() * (s.M + size)) {}
    static int64_t bytes(const Shape &s, int64_t size) { return s.rows() * (s.M + 2 * size); }
    uint8_t *codes = nullptr;
    void *bias = nullptr, *scale = nullptr;
};

// Whether the combine of the gradient rows adds the gate's share of the gradient of x (planmoe_layer_dx): up to 8 experts always.  Beyond, the other way is
// the combine, a cast and the library's product with a reduction of as many as there are experts, and one pass reads 16 weights a value from L2.
// us, 16 experts, one pass and the other way:
//   bf16         64 x 1024 5.9, 11.2    4096 x 1024 11.2, 19.8    16384 x 1024 39.8, 41.3    1024 x 4096 14.0, 18.9    16384 x 4096 142, 143
//   bf16, int8   64 x 1024 6.7, 12.1    4096 x 2048 26.5, 30.6    16384 x 1024 52.1, 44.7    1024 x 4096 18.0, 20.6    4096 x 4096 52.2, 45.4
//   fp32         1024 x 256 4.9, 7.3    4096 x 1024 13.4, 21.4    16384 x 2048 81, 125
//   fp32, int8   1024 x 256 7.0, 8.0    1024 x 1024 14.6, 12.4    4096 x 1024 19.8, 25.5     16384 x 2048 124, 132
// (fp32, fewer tokens and rows above 2 KB: one pass would be the faster one here too, 64 x 1024 4.2 and 7.0, but it rounds the sum once an expert where the other way adds the gate's
// whole product: error against 64 bits 1.0e-7 of the norm, and 3.8e-8.)
bool dx_in_one(const Shape &s, int codec)
{
    if (s.E <= 8) return true;
    const int64_t values = (int64_t)s.T * s.M;
    if (s.E > 16 || (int64_t)s.M * (s.dt == PLANMOE_F32 ? 4 : 2) > 8192) return false;
    if (s.dt == PLANMOE_F32) return s.M <= 512 || s.T >= 4096 || (s.T >= 1024 && codec != CODEC_INT8);
    return codec != CODEC_INT8 || (s.T <= 8192 && values <= (1 << 23));
}

// The second product and the combine, without a codec or through the int8 codec; kept: its codes, keep: the rows without it, for a backward pass
void product_combine(const Shape &s, int codec, const void *h, const Tensor &w2, const Tensor &b2, const float *gates, const int32_t *idx, const int32_t *loc,
                     const int32_t *cnt, void *ye, bool keep, const Kept &kept, const Tensor &y, void *shares_at, size_t shares, void *st)
{
    const int coded = codec == CODEC_INT8;
    if (shares > 0) {
        PM_CALL(planmoe_layer_product_combine(h, w2.data_ptr(), b2.data_ptr(), s.dt, coded, s.H, gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, cnt, 1, s.hint(), ye,
                                              keep, kept.codes, kept.bias, kept.scale, y.data_ptr(), shares_at, shares, st));
        return;
    }
    PM_CALL(planmoe_expert_gemm(0, s.dt, h, w2.data_ptr(), b2.data_ptr(), 0, s.E, s.cap, s.M, s.H, cnt, s.k, 1, s.hint(), ye, st));
    if (kept.codes) PM_CALL(planmoe_layer_combine_keep(ye, s.dt, gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, y.data_ptr(), kept.codes, kept.bias, kept.scale, st));
    else PM_CALL(planmoe_layer_combine(ye, s.dt, coded, gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, y.data_ptr(), st));
}

Pass forward_pass(const Tensor &x, const Tensor &wg, const Tensor &w1, const Tensor &b1, const Tensor &w2, const Tensor &b2, const Shape &s,
                  bool fp32_gate, bool normalize, int codec, bool keep)
{
    void *st = current_stream();
    Pass p;
    const auto score_type = fp32_gate ? at::kFloat : x.scalar_type();
    p.r = Routing(s, score_type);
    p.r.lie_in(at::empty({p.r.words}, x.options().dtype(at::kInt)));
    p.l_aux = at::empty({}, x.options().dtype(at::kFloat));
    const int64_t ws_bytes = ((int64_t)planmoe_forward_workspace_bytes(s.T, s.E, s.k) + 255) / 256 * 256;
    const size_t shares = s.shares(codec);
    Tensor ws = bytes(ws_bytes + (int64_t)shares, x);
    int32_t *idx = p.r.idx, *loc = p.r.loc, *cnt = p.r.cnt;
    void *const scores = keep ? p.r.scores : nullptr;
    if (codec == CODEC_ZFP) {
        PM_CALL(planmoe_gate_route(x.data_ptr(), wg.data_ptr(), s.dt, fp32_gate, nullptr, s.T, s.M, s.E, s.k, normalize, idx, loc, p.r.gates,
                                   s.T, nullptr, scores, p.l_aux.data_ptr<float>(), cnt, ws.data_ptr(), (size_t)ws.numel(), st));
        p.xe = at::empty({s.rows(), s.M}, x.options());
        ws = zfp_workspace(s, x);
        PM_CALL(planmoe_layer_zfp_dispatch(floats(x), idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, cnt, p.xe.data_ptr<float>(), ws.data_ptr(),
                                           (size_t)ws.numel(), st));
    } else if (codec == CODEC_LZ) {
        p.xe = at::empty({s.rows(), s.M}, x.options());
        PM_CALL(planmoe_forward_plain(x.data_ptr(), wg.data_ptr(), s.dt, fp32_gate, nullptr, s.T, s.M, s.E, s.k, normalize, s.cap, idx, loc,
                                      p.r.gates, s.T, nullptr, scores, p.l_aux.data_ptr<float>(), cnt, p.xe.data_ptr(), ws.data_ptr(),
                                      (size_t)ws.numel(), st));
        p.xe = lz_round_trip(p.xe, st);
    } else {
        p.xe = at::empty({s.rows(), s.M}, x.options());
        PM_CALL(planmoe_layer_dispatch(x.data_ptr(), wg.data_ptr(), s.dt, fp32_gate, nullptr, s.T, s.M, s.E, s.k, normalize, s.cap, codec, idx, loc,
                                       p.r.gates, s.T, scores, p.l_aux.data_ptr<float>(), cnt, p.xe.data_ptr(), ws.data_ptr(),
                                       (size_t)ws.numel(), st));
    }
    const Live live = live_rows(p, s, codec);
    p.h = at::empty({s.rows(), s.H}, x.options());
    PM_CALL(planmoe_expert_gemm(0, s.dt, p.xe.data_ptr(), w1.data_ptr(), b1.data_ptr(), 1, s.E, s.cap, s.H, s.M, live.counts, live.planes, live.round,
                                s.hint(), p.h.data_ptr(), st));
    p.ye = at::empty({s.rows(), s.M}, x.options());
    p.y = at::empty({s.T, s.M}, x.options());
    Tensor wide;
    const float *const gates = p.r.float_gates(s, wide);
    if (codec == CODEC_NONE || codec == CODEC_INT8) {
        Kept kept;
        if (codec == CODEC_INT8 && keep) {
            // (the backward pass reads the codes: a byte a value is held until then, as between Compress and its backward)
            p.codes = bytes(Kept::bytes(s, x.element_size()), x);
            kept = Kept(p.codes, s, x.element_size());
        }
        product_combine(s, codec, p.h.data_ptr(), w2, b2, gates, idx, loc, cnt, p.ye.data_ptr(), keep, kept, p.y, ws.data_ptr<uint8_t>() + ws_bytes, shares, st);
        if (p.codes.defined()) p.ye = Tensor();
        return p;
    }
    PM_CALL(planmoe_expert_gemm(0, s.dt, p.h.data_ptr(), w2.data_ptr(), b2.data_ptr(), 0, s.E, s.cap, s.M, s.H, live.counts, live.planes, live.round,
                                s.hint(), p.ye.data_ptr(), st));
    if (codec == CODEC_ZFP) {
        if (keep) p.stream = zfp_stream(s, x);
        zfp_rows(p.ye.data_ptr(), p.stream, p, s, st);
    }
    if (codec == CODEC_LZ) p.ye = lz_round_trip(p.ye, st);
    PM_CALL(planmoe_layer_combine(p.ye.data_ptr(), s.dt, 0, gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, p.y.data_ptr(), st));
    if (p.stream.defined()) p.ye = Tensor();         // (the backward pass reads the stream)
    return p;
}

// A pass that nothing is kept of: what only its launches see lies in one buffer (eight allocations take the host 9 us, a third
// of a decode step's time, three 3).  The lz codec has its own buffers.  The products are those of a pass that a backward pass follows: the
// same bits with and without autograd (a checkpoint's first run is without, its second with).
std::tuple<Tensor, Tensor> inference_pass(const Tensor &x, const Tensor &wg, const Tensor &w1, const Tensor &b1, const Tensor &w2, const Tensor &b2,
                                          const Shape &s, bool fp32_gate, bool normalize, int codec)
{
    void *st = current_stream();
    const int64_t size = x.element_size();
    int64_t end = 0;
    auto piece = [&](int64_t n) { const int64_t at = end; end += (n + 255) / 256 * 256; return at; };
    const bool bf16_gate = !fp32_gate && s.dt != PLANMOE_F32;
    const size_t ws_bytes = std::max(planmoe_forward_workspace_bytes(s.T, s.E, s.k), codec == CODEC_ZFP ? planmoe_layer_zfp_workspace_bytes(s.E, s.cap) : 0);
    const int64_t idx_at = piece((int64_t)s.k * s.T * 4), loc_at = piece((int64_t)s.k * s.T * 4), cnt_at = piece((int64_t)s.k * s.E * 4),
                  gates_at = piece((int64_t)s.k * s.T * (bf16_gate ? size : 4)), wide_at = bf16_gate ? piece((int64_t)s.k * s.T * 4) : 0,
                  ws_at = piece((int64_t)ws_bytes), xe_at = piece(s.rows() * s.M * size), h_at = piece(s.rows() * s.H * size), ye_at = piece(s.rows() * s.M * size);
    const size_t shares = s.shares(codec);
    const int64_t shares_at = piece((int64_t)shares);
    const Tensor pool = bytes(end, x);
    uint8_t *const base = pool.data_ptr<uint8_t>();
    int32_t *const idx = (int32_t *)(base + idx_at), *const loc = (int32_t *)(base + loc_at), *const cnt = (int32_t *)(base + cnt_at);
    void *const ws = base + ws_at, *const xe = base + xe_at, *const h = base + h_at, *const ye = base + ye_at;
    const float *gates = (const float *)(base + gates_at);
    Tensor l_aux = at::empty({}, x.options().dtype(at::kFloat)), y = at::empty({s.T, s.M}, x.options());
    if (codec == CODEC_ZFP) {
        PM_CALL(planmoe_gate_route(x.data_ptr(), wg.data_ptr(), s.dt, fp32_gate, nullptr, s.T, s.M, s.E, s.k, normalize, idx, loc, base + gates_at, s.T, nullptr,
                                   nullptr, l_aux.data_ptr<float>(), cnt, ws, ws_bytes, st));
        PM_CALL(planmoe_layer_zfp_dispatch(floats(x), idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, cnt, (float *)xe, ws, ws_bytes, st));
    } else {
        PM_CALL(planmoe_layer_dispatch_product(x.data_ptr(), wg.data_ptr(), s.dt, fp32_gate, s.T, s.M, s.E, s.k, normalize, s.cap, codec, idx, loc, base + gates_at,
                                               s.T, l_aux.data_ptr<float>(), cnt, w1.data_ptr(), b1.data_ptr(), s.H, s.hint(), xe, h, ws, ws_bytes, st));
    }
    if (bf16_gate) {
        at::from_blob(base + wide_at, {s.k, s.T}, x.options().dtype(at::kFloat)).copy_(at::from_blob(base + gates_at, {s.k, s.T}, x.options()));
        gates = (const float *)(base + wide_at);
    }
    if (codec != CODEC_ZFP) {
        product_combine(s, codec, h, w2, b2, gates, idx, loc, cnt, ye, false, Kept{}, y, base + shares_at, shares, st);
        return {y, l_aux};
    }
    PM_CALL(planmoe_expert_gemm(0, s.dt, xe, w1.data_ptr(), b1.data_ptr(), 1, s.E, s.cap, s.H, s.M, cnt, s.k, 4, s.hint(), h, st));
    PM_CALL(planmoe_expert_gemm(0, s.dt, h, w2.data_ptr(), b2.data_ptr(), 0, s.E, s.cap, s.M, s.H, cnt, s.k, 4, s.hint(), ye, st));
    PM_CALL(planmoe_layer_zfp_rows((float *)ye, s.M, s.E, s.cap, cnt, s.k, nullptr, 0, st));
    PM_CALL(planmoe_layer_combine(ye, s.dt, 0, gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, y.data_ptr(), st));
    return {y, l_aux};
}

Shape shape_of(const Tensor &x, const Tensor &wg, const Tensor &w1, int64_t k, int64_t cap)
{
    Shape s;
    s.T = (int)x.size(0);
    s.M = (int)x.size(1);
    s.E = (int)wg.size(0);
    s.H = (int)w1.size(2);
    s.k = (int)k;
    s.cap = (int)cap;
    s.dt = pm_dtype(x.scalar_type());
    return s;
}

void check(const Tensor &x, const Tensor &wg, const Tensor &w1, const Tensor &b1, const Tensor &w2, const Tensor &b2, int64_t k, int64_t cap)
{
    TORCH_CHECK(x.dim() == 2 && wg.dim() == 2 && w1.dim() == 3 && w2.dim() == 3 && b1.dim() == 2 && b2.dim() == 2, "ffn_layer: wrong ranks");
    const int64_t M = x.size(1), E = wg.size(0), H = w1.size(2);
    TORCH_CHECK(wg.size(1) == M && w1.size(0) == E && w1.size(1) == M && w2.size(0) == E && w2.size(1) == H && w2.size(2) == M &&
                b1.size(0) == E && b1.size(1) == H && b2.size(0) == E && b2.size(1) == M, "ffn_layer: shapes do not fit");
    TORCH_CHECK(k >= 1 && k <= E && cap >= 1 && x.size(0) >= 1, "ffn_layer: bad routing shape");
    for (const Tensor *t : {&x, &wg, &w1, &b1, &w2, &b2})
        TORCH_CHECK(t->is_cuda() && t->is_contiguous() && t->scalar_type() == x.scalar_type() && t->device() == x.device(),
                    "ffn_layer: contiguous GPU tensors of one dtype on one device");
}

struct FfnLayer : public torch::autograd::Function<FfnLayer> {
    static torch::autograd::variable_list forward(torch::autograd::AutogradContext *ctx, const Tensor &x, const Tensor &wg, const Tensor &w1,
                                                  const Tensor &b1, const Tensor &w2, const Tensor &b2, int64_t k, int64_t cap, bool fp32_gate,
                                                  bool normalize, int64_t codec)
    {
        const Shape s = shape_of(x, wg, w1, k, cap);
        Pass p = forward_pass(x, wg, w1, b1, w2, b2, s, fp32_gate, normalize, (int)codec, true);
        ctx->save_for_backward({x, wg, w1, w2, p.r.held, p.xe, p.h, codec == CODEC_ZFP ? p.stream : codec == CODEC_INT8 ? p.codes : p.ye});
        ctx->saved_data["form"] = std::vector<int64_t>{k, cap, normalize, codec, fp32_gate};
        ctx->set_materialize_grads(false);
        return {p.y, p.l_aux};
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &wg = saved[1], &w1 = saved[2], &w2 = saved[3];
        const c10::DeviceGuard guard(x.device());
        const std::vector<int64_t> form = ctx->saved_data["form"].toIntVector();
        const int codec = (int)form[3];
        const bool normalize = form[2] != 0;
        const Shape s = shape_of(x, wg, w1, form[0], form[1]);
        void *st = current_stream();
        Pass p;
        p.r = Routing(s, form[4] ? at::kFloat : x.scalar_type());
        p.r.lie_in(saved[4]);
        p.xe = saved[5];
        p.h = saved[6];
        const Tensor &ye = saved[7];                 // (the rows; zfp: their stream; int8: their codes)
        const int32_t *idx = p.r.idx, *loc = p.r.loc;
        const auto score_options = x.options().dtype(p.r.type);
        const bool need_x = ctx->needs_input_grad(0), need_gate = ctx->needs_input_grad(1), need_w1 = ctx->needs_input_grad(2),
                   need_b1 = ctx->needs_input_grad(3), need_w2 = ctx->needs_input_grad(4), need_b2 = ctx->needs_input_grad(5);
        Tensor dx, dwg, dw1, db1, dw2, db2, grad_gates, gf;
        bool gate_added = false;                     // (dx has the gate's share)
        Tensor gl = grads[1].defined() ? grads[1].to(at::kFloat).contiguous() : Tensor();
        const float *dl = gl.defined() ? floats(gl) : nullptr;
        const int32_t *count0 = gl.defined() ? p.r.cnt : nullptr;
        // the logits' gradient, in the scores' precision
        auto route_bwd = [&]() {
            Tensor gg = grad_gates.defined() ? grad_gates.to(p.r.type) : at::zeros({s.k, s.T}, score_options);
            Tensor g = at::empty({s.T, s.E}, score_options);
            PM_CALL(planmoe_route_bwd(p.r.scores, pm_dtype(p.r.type), idx, gg.data_ptr(), s.T, s.T, s.E, s.k, normalize, dl, count0, 1,
                                      g.data_ptr(), st));
            return g;
        };
        auto as_float = [](const Tensor &g) { return g.scalar_type() == at::kFloat ? g : g.to(at::kFloat); };
        // everything is asked for, as in a training step: reductions share their launches, and the gate's part of dx is added in the combine
        const bool whole = grads[0].defined() && need_x && need_gate && need_w1 && need_b1 && need_w2 && need_b2;
        if (grads[0].defined()) {
            const Tensor grad = as_rows(grads[0]);
            Tensor wide;
            const float *const gates = p.r.float_gates(s, wide);
            const Live live = live_rows(p, s, codec);
            const bool logits = whole && s.k <= 64 && (codec == CODEC_NONE || codec == CODEC_INT8);
            // what only this pass sees; with everything asked for in one buffer
            const int64_t size = x.element_size(), wide_rows = s.rows() * s.M * size, hidden_rows = s.rows() * s.H * size;
            const int64_t sums_bytes = whole ? (int64_t)planmoe_layer_sums_workspace_bytes(s.E, s.cap, s.T, s.M) : 0;
            const int64_t db1_bytes = need_b1 ? (int64_t)planmoe_expert_gemm_relu_bwd_workspace_bytes(s.E, s.cap, s.H) : 0;
            auto room = [](int64_t n) { return (n + 255) / 256 * 256; };
            Tensor pool, alone[5];
            int64_t used = 0;
            int count = 0;
            if (whole && codec != CODEC_LZ) pool = bytes(2 * room(wide_rows) + room(hidden_rows) + room(sums_bytes) + room(db1_bytes), x);
            auto scratch = [&](int64_t n) -> void * {
                if (!pool.defined()) return (alone[count++] = bytes(n, x)).data_ptr();
                used += room(n);
                return pool.data_ptr<uint8_t>() + used - room(n);
            };
            (logits ? gf : grad_gates) = at::empty({logits ? s.T : s.k, logits ? s.E : s.T}, x.options().dtype(at::kFloat));
            Tensor coded_rows;                       // (lz)
            void *gye, *sums = nullptr;
            if (codec == CODEC_ZFP) {
                gye = scratch(wide_rows);
                Tensor ws = zfp_workspace(s, x);
                PM_CALL(planmoe_layer_zfp_combine_bwd(ye.data_ptr(), floats(grad), gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, p.r.cnt,
                                                      (float *)gye, grad_gates.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), st));
            } else if (codec == CODEC_LZ) {
                Tensor buf = at::empty({s.rows(), s.M}, x.options()), ws = bytes((int64_t)planmoe_dispatch_workspace_bytes(s.E, s.cap), x);
                PM_CALL(planmoe_combine_bwd(grad.data_ptr(), ye.data_ptr(), s.dt, gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, buf.data_ptr(),
                                            grad_gates.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), st));
                coded_rows = lz_round_trip(buf, st);
                gye = coded_rows.data_ptr();
            } else {
                gye = scratch(wide_rows);
                if (logits) {
                    const bool coded = codec == CODEC_INT8;
                    const Kept kept = coded ? Kept(ye, s, x.element_size()) : Kept{};
                    PM_CALL(planmoe_layer_combine_bwd_logits(grad.data_ptr(), coded ? kept.codes : ye.data_ptr(), kept.bias, kept.scale, s.dt, coded,
                                                             gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, gye, p.r.scores,
                                                             pm_dtype(p.r.type), normalize, dl, count0, gf.data_ptr<float>(), st));
                } else if (codec == CODEC_INT8) {
                    const Kept kept(ye, s, x.element_size());
                    PM_CALL(planmoe_layer_combine_bwd_codes(grad.data_ptr(), kept.codes, kept.bias, kept.scale, s.dt, gates, idx, loc, s.T, s.k,
                                                            s.T, s.M, s.E, s.cap, gye, grad_gates.data_ptr<float>(), st));
                } else {
                    PM_CALL(planmoe_layer_combine_bwd(grad.data_ptr(), ye.data_ptr(), s.dt, 0, gates, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap,
                                                      gye, grad_gates.data_ptr<float>(), st));
                }
            }
            if (whole) {
                if (!gf.defined()) gf = as_float(route_bwd());
                sums = scratch(sums_bytes);
                PM_CALL(planmoe_layer_sums(gye, s.dt, s.E, s.cap, live.counts, live.planes, live.round, x.data_ptr(), floats(gf), s.T, s.M,
                                           sums, (size_t)sums_bytes, st));
                db2 = at::empty({s.E, s.M}, x.options());
                dwg = at::empty_like(wg);
            }
            auto colsum = [&](const void *a, int cols) {
                Tensor out = at::empty({s.E, cols}, x.options()), ws = bytes((int64_t)planmoe_rows_colsum_workspace_bytes(s.E, s.cap, cols), x);
                PM_CALL(planmoe_rows_colsum(a, s.dt, s.E, s.cap, cols, live.counts, live.planes, live.round, out.data_ptr(), ws.data_ptr(),
                                            (size_t)ws.numel(), st));
                return out;
            };
            if (need_w2) {
                dw2 = at::empty_like(w2);
                PM_CALL(planmoe_expert_gemm(2, s.dt, p.h.data_ptr(), gye, nullptr, 0, s.E, s.H, s.M, s.cap, live.counts, live.planes, live.round,
                                            s.hint(), dw2.data_ptr(), st));
            }
            if (need_b2 && !whole) db2 = colsum(gye, s.M);
            if (need_x || need_w1 || need_b1) {
                void *const gh = scratch(hidden_rows), *const ws = need_b1 ? scratch(db1_bytes) : nullptr;
                if (need_b1) db1 = at::empty({s.E, s.H}, x.options());
                if (whole)
                    PM_CALL(planmoe_layer_relu_bwd(s.dt, gye, w2.data_ptr(), p.h.data_ptr(), s.E, s.cap, s.H, s.M, live.counts, live.planes,
                                                   live.round, s.hint(), gh, raw(db1), ws, (size_t)db1_bytes, sums,
                                                   (size_t)sums_bytes, s.T, raw(db2), raw(dwg), st));
                else
                    PM_CALL(planmoe_expert_gemm_relu_bwd(s.dt, gye, w2.data_ptr(), p.h.data_ptr(), s.E, s.cap, s.H, s.M, live.counts, live.planes,
                                                         live.round, s.hint(), gh, raw(db1), ws, (size_t)db1_bytes, st));
                if (need_w1) {
                    dw1 = at::empty_like(w1);
                    PM_CALL(planmoe_expert_gemm(2, s.dt, p.xe.data_ptr(), gh, nullptr, 0, s.E, s.M, s.H, s.cap, live.counts, live.planes,
                                                live.round, s.hint(), dw1.data_ptr(), st));
                }
                if (need_x) {
                    Tensor lz_rows = codec == CODEC_LZ ? at::empty({s.rows(), s.M}, x.options()) : Tensor();
                    void *gxe = codec == CODEC_LZ ? lz_rows.data_ptr() : scratch(wide_rows);
                    PM_CALL(planmoe_expert_gemm(1, s.dt, gh, w1.data_ptr(), nullptr, 0, s.E, s.cap, s.M, s.H, live.counts, live.planes, live.round,
                                                s.hint(), gxe, st));
                    if (codec == CODEC_ZFP) zfp_rows(gxe, Tensor(), p, s, st);
                    if (codec == CODEC_LZ) gxe = (lz_rows = lz_round_trip(lz_rows, st)).data_ptr();
                    dx = at::empty_like(x);
                    if (whole && dx_in_one(s, codec)) {
                        PM_CALL(planmoe_layer_dx(gxe, s.dt, codec == CODEC_INT8, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, floats(gf),
                                                 wg.data_ptr(), dx.data_ptr(), st));
                        return {dx, dwg, dw1, db1, dw2, db2, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
                    }
                    if (s.E > 8 && dx_in_one(s, codec)) {
                        if (!gf.defined()) gf = as_float(route_bwd());
                        PM_CALL(planmoe_layer_dx(gxe, s.dt, codec == CODEC_INT8, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap, floats(gf),
                                                 wg.data_ptr(), dx.data_ptr(), st));
                        gate_added = true;
                    } else {
                        PM_CALL(planmoe_layer_combine(gxe, s.dt, codec == CODEC_INT8, nullptr, idx, loc, s.T, s.k, s.T, s.M, s.E, s.cap,
                                                      dx.data_ptr(), st));
                    }
                }
            }
        }
        // gates and loss back through the routing into the gate's weight and x
        if ((grad_gates.defined() || gf.defined() || grads[1].defined()) && (need_x || need_gate)) {
            if (!gf.defined()) gf = as_float(route_bwd());
            if (need_gate && !dwg.defined()) {
                dwg = at::empty_like(wg);
                Tensor ws = bytes((int64_t)planmoe_gate_dw_workspace_bytes(s.T, s.M, s.E), x);
                PM_CALL(planmoe_gate_dw(x.data_ptr(), s.dt, floats(gf), s.T, s.M, s.E, dwg.data_ptr(), ws.data_ptr(), (size_t)ws.numel(), st));
            }
            if (need_x && !gate_added) {
                if (!dx.defined()) {
                    dx = at::mm(gf.to(x.scalar_type()), wg);
                } else if (s.E <= 8) {
                    PM_CALL(planmoe_gate_dx_accumulate(dx.data_ptr(), s.dt, floats(gf), wg.data_ptr(), s.T, s.M, s.E, st));
                } else {
                    dx.addmm_(gf.to(x.scalar_type()), wg);
                }
            }
        }
        return {dx, dwg, dw1, db1, dw2, db2, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// (y [T, M], l_aux fp32); codec: 0 none, 1 int8, 2 zfp, 3 lz
std::tuple<Tensor, Tensor> ffn_layer(const Tensor &x, const Tensor &wg, const Tensor &w1, const Tensor &b1, const Tensor &w2, const Tensor &b2,
                                     int64_t k, int64_t cap, bool fp32_gate, bool normalize, int64_t codec)
{
    check(x, wg, w1, b1, w2, b2, k, cap);
    const c10::DeviceGuard guard(x.device());
    // (a forward-mode tangent goes to the node as well, which refuses it: it would be lost here without a word)
    bool grad = false;
    for (const Tensor *t : {&x, &wg, &w1, &b1, &w2, &b2}) grad |= (at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(0).defined();
    if (!grad) {
        const at::NoGradGuard no_grad;
        if (codec != CODEC_LZ) return inference_pass(x, wg, w1, b1, w2, b2, shape_of(x, wg, w1, k, cap), fp32_gate, normalize, (int)codec);
        Pass p = forward_pass(x, wg, w1, b1, w2, b2, shape_of(x, wg, w1, k, cap), fp32_gate, normalize, (int)codec, false);
        return {p.y, p.l_aux};
    }
    auto out = FfnLayer::apply(x, wg, w1, b1, w2, b2, k, cap, fp32_gate, normalize, codec);
    return {out[0], out[1]};
}

} // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    pybind11::register_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const Failure &e) {
            PyErr_SetString(pybind11::module_::import("planmoe_amd._lib").attr("PlanMoEError").ptr(), e.what());
        }
    });
    def_routing(m);
    m.def("ffn_layer", &ffn_layer, pybind11::call_guard<pybind11::gil_scoped_release>(), "the layer with its built-in experts, forward (and its autograd node)");
}
