// The functional routing API's host side (fast_dispatch.py:16-79, 140-207): extract_critical, fast_encode and
// fast_decode with their gradients, one call and one autograd node each.
//
// Driven step by step from Python a pass forward and backward took 370 us of host time for 225 us (8192 x 2048
// fp32) or 124 us (3001 x 1030 fp16) of GPU time, and its 22 - 25 launches were half torch's own: zeros in place
// of the gradients that integer outputs never have, and a gradient of the whole [k, T] plane, with a
// copy and an addition, for every choice that was a view of it.  Here every choice's gates are an output of
// the node, laid out as planes of one buffer, and gradients that come back as planes are taken as they lie.
#include "host.hpp"

namespace {

using namespace planmoe_host;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// part of a flat buffer as a tensor of its own: no view in autograd's sense (an output of a node may be one), its in-place
// changes are counted apart from the buffer's
Tensor piece(const Tensor &base, int64_t first, int64_t size)
{
    const at::AutoDispatchBelowADInplaceOrView guard;
    return base.narrow(0, first, size);
}

// k flat tensors as planes of one buffer, equally far apart: the distance in elements (0: any, one plane), or -1
int64_t spacing(const std::vector<Tensor> &t)
{
    if (t.size() == 1) return 0;
    const int64_t d = (const char *)t[1].data_ptr() - (const char *)t[0].data_ptr(), size = t[0].element_size();
    if (d < t[0].numel() * size || d % size) return -1;
    for (size_t j = 1; j < t.size(); ++j)
        if ((const char *)t[j].data_ptr() - (const char *)t[0].data_ptr() != (int64_t)j * d || !t[j].storage().is_alias_of(t[0].storage())) return -1;
    return d / size;
}

bool flat(const std::vector<Tensor> &t, size_t k, int64_t n, at::ScalarType type, const Tensor &data)
{
    if (t.size() != k) return false;
    for (const Tensor &v : t)
        if (!v.is_cuda() || v.device() != data.device() || v.dim() != 1 || v.numel() != n || v.scalar_type() != type || !v.is_contiguous()) return false;
    return true;
}

struct Planes {
    std::vector<Tensor> idx, loc, gates;         // (what keeps the memory)
    const int32_t *i() const { return ints(idx[0]); }
    const int32_t *l() const { return ints(loc[0]); }
    const float *g() const { return gates.empty() ? nullptr : floats(gates[0]); }
    int64_t stride, samples;
    int k, experts, capacity;
};

Planes planes_of(std::vector<Tensor> idx, std::vector<Tensor> loc, std::vector<Tensor> gates, int experts, int capacity)
{
    Planes p;
    p.k = (int)idx.size();
    p.samples = idx[0].numel();
    p.experts = experts;
    p.capacity = capacity;
    const int64_t a = spacing(idx), b = spacing(loc), c = gates.empty() ? a : spacing(gates);
    if (a < 0 || a != b || a != c) {
        const at::NoGradGuard no_grad;
        idx = {at::stack(idx)};
        loc = {at::stack(loc)};
        if (!gates.empty()) gates = {at::stack(gates)};
    }
    p.stride = a > 0 && a == b && a == c ? a : p.samples;
    p.idx = std::move(idx);
    p.loc = std::move(loc);
    p.gates = std::move(gates);
    return p;
}

Tensor scatter(const Tensor &x, const float *gates, const Planes &p)
{
    const int64_t M = x.size(-1);
    Tensor out = at::empty({p.experts, p.capacity, M}, x.options()), ws = bytes((int64_t)planmoe_dispatch_workspace_bytes(p.experts, p.capacity), x);
    PM_CALL(planmoe_dispatch_fwd(x.data_ptr(), pm_dtype(x.scalar_type()), gates, p.i(), p.l(), p.stride, p.k, (int)p.samples, (int)M, p.experts, p.capacity,
                                 out.data_ptr(), ws.data_ptr(), (size_t)ws.numel(), current_stream()));
    return out;
}

Tensor gather(const Tensor &slots, const float *gates, const Planes &p)
{
    const int64_t M = slots.size(-1);
    Tensor out = at::empty({p.samples, M}, slots.options());
    PM_CALL(planmoe_combine_fwd(slots.data_ptr(), pm_dtype(slots.scalar_type()), gates, p.i(), p.l(), p.stride, p.k, (int)p.samples, (int)M, p.capacity,
                                out.data_ptr(), current_stream()));
    return out;
}

std::vector<Tensor> planes_as_tensors(const Tensor &buffer, const Planes &p)
{
    std::vector<Tensor> parts;
    for (int j = 0; j < p.k; ++j) parts.push_back(piece(buffer, j * p.stride, p.samples));
    return parts;
}

// <slots[slot_j], x[t]>, one tensor a choice, planes of one buffer
std::vector<Tensor> gate_gradients(const Tensor &x, const Tensor &slots, const Planes &p)
{
    Tensor out = at::empty({p.k * p.stride}, x.options().dtype(at::kFloat));
    PM_CALL(planmoe_bwd_gate(x.data_ptr(), slots.data_ptr(), pm_dtype(x.scalar_type()), p.i(), p.l(), p.stride, p.k, (int)p.samples, (int)x.size(-1),
                             p.capacity, out.data_ptr<float>(), current_stream()));
    return planes_as_tensors(out, p);
}

// both gradients of a gather, in one pass over what comes back
std::tuple<Tensor, std::vector<Tensor>> gather_backward(const Tensor &grad, const Tensor &slots, const Planes &p)
{
    const int64_t M = grad.size(-1);
    Tensor out = at::empty({p.experts, p.capacity, M}, grad.options()), ws = bytes((int64_t)planmoe_dispatch_workspace_bytes(p.experts, p.capacity), grad);
    Tensor gg = at::empty({p.k * p.stride}, grad.options().dtype(at::kFloat));
    PM_CALL(planmoe_combine_bwd(grad.data_ptr(), slots.data_ptr(), pm_dtype(grad.scalar_type()), p.g(), p.i(), p.l(), p.stride, p.k, (int)p.samples, (int)M,
                                p.experts, p.capacity, out.data_ptr(), gg.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), current_stream()));
    return {out, planes_as_tensors(gg, p)};
}

// encode (tokens to slots) and decode (slots to tokens); each is the other's backward pass
template <bool ENCODE>
struct Move : public torch::autograd::Function<Move<ENCODE>> {
    static Tensor forward(AutogradContext *ctx, const Tensor &data, at::TensorList gates, Planes *planes, Planes *given)
    {
        ctx->set_materialize_grads(false);
        ctx->saved_data["planes"] = c10::IValue::make_capsule(c10::make_intrusive<Held>(*given));
        if (!gates.empty()) ctx->saved_data["data"] = data;         // (for the gates' gradient)
        ctx->saved_data["sizes"] = data.sizes().vec();
        return ENCODE ? scatter(data, planes->g(), *planes) : gather(data, planes->g(), *planes);
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const Planes &kept = static_cast<Held *>(ctx->saved_data["planes"].toCapsule().get())->planes;
        const int gates = (int)kept.gates.size();
        variable_list out(3 + gates);
        if (!grads[0].defined()) return out;
        const Tensor grad = grads[0].contiguous();
        const c10::DeviceGuard guard(grad.device());
        // (looked at again: what the planes lie in may have been exchanged since the forward pass)
        TORCH_CHECK(flat(kept.idx, kept.k, kept.samples, at::kInt, grad) && flat(kept.loc, kept.k, kept.samples, at::kInt, grad) &&
                    (gates == 0 || flat(kept.gates, kept.k, kept.samples, at::kFloat, grad)), "the routing's tensors have changed their shape, type or device");
        const Planes p = planes_of(kept.idx, kept.loc, kept.gates, kept.experts, kept.capacity);
        bool to_gates = false;
        for (int j = 0; j < gates; ++j) to_gates |= ctx->needs_input_grad(1 + j);
        const Tensor data = to_gates ? ctx->saved_data["data"].toTensor() : Tensor();
        Tensor d;
        std::vector<Tensor> g;
        if (!ENCODE && to_gates && ctx->needs_input_grad(0)) {
            std::tie(d, g) = gather_backward(grad, data, p);
        } else {
            if (ctx->needs_input_grad(0)) d = ENCODE ? gather(grad, p.g(), p) : scatter(grad, p.g(), p);
            if (to_gates) g = ENCODE ? gate_gradients(data, grad, p) : gate_gradients(grad, data, p);
        }
        if (d.defined()) out[0] = d.view(ctx->saved_data["sizes"].toIntVector());
        for (size_t j = 0; j < g.size(); ++j) out[1 + j] = g[j];
        return out;
    }

    struct Held : torch::CustomClassHolder {
        explicit Held(Planes p) : planes(std::move(p)) {}
        Planes planes;
    };
};

// None where the arguments are not what the kernels take as they are (the caller converts them, or says what is wrong)
template <bool ENCODE>
std::optional<Tensor> move(const Tensor &data_, const std::vector<Tensor> &gates, const std::vector<Tensor> &idx, const std::vector<Tensor> &loc,
                           int64_t experts, int64_t capacity)
{
    if (!data_.is_cuda() || !pm_dtype_ok(data_.scalar_type()) || data_.dim() < 2 || idx.empty() || !idx[0].defined()) return std::nullopt;
    const size_t k = idx.size();
    const int64_t n = idx[0].numel(), M = data_.size(-1);
    if (n < 1 || M < 1 || experts < 1 || capacity < 1 || experts * capacity >= ((int64_t)1 << 31) || (int64_t)k * n >= ((int64_t)1 << 31)) return std::nullopt;
    if (ENCODE ? data_.dim() != 2 || data_.size(0) != n : data_.numel() != experts * capacity * M) return std::nullopt;
    if (!flat(idx, k, n, at::kInt, data_) || !flat(loc, k, n, at::kInt, data_) || !(gates.empty() || flat(gates, k, n, at::kFloat, data_))) return std::nullopt;
    const c10::DeviceGuard guard(data_.device());
    const Tensor data = data_.contiguous();
    Planes p = planes_of(idx, loc, gates, (int)experts, (int)capacity), given = p;
    given.idx = idx;
    given.loc = loc;
    given.gates = gates;
    return Move<ENCODE>::apply(data, at::TensorList(gates), &p, &given);
}

// ------------------------------------------------------------------ routing
struct Routed {
    int T, E, k;
    bool normalize, want_loss;
    Tensor read;                                 // what the backward pass reads: indices [k T], counts [k E]
    std::vector<Tensor> locations;
};

struct Route : public torch::autograd::Function<Route> {
    static variable_list forward(AutogradContext *ctx, const Tensor &scores, Routed *r)
    {
        ctx->set_materialize_grads(false);
        const int64_t plane = (int64_t)r->k * r->T, read = plane + (int64_t)r->k * r->E;
        Tensor ints_ = at::empty({read + plane}, scores.options().dtype(at::kInt)), gates = at::empty({plane}, scores.options());
        Tensor loss = r->want_loss ? at::empty({}, scores.options().dtype(at::kFloat)) : Tensor();
        Tensor ws = bytes((int64_t)planmoe_route_workspace_bytes(r->T, r->E, r->k), scores);
        int32_t *i = ints_.data_ptr<int32_t>();
        PM_CALL(planmoe_route_topk(scores.data_ptr(), pm_dtype(scores.scalar_type()), 0, nullptr, r->T, r->E, r->k, r->normalize, i, i + read,
                                   gates.data_ptr(), r->T, nullptr, loss.defined() ? loss.data_ptr<float>() : nullptr, i + plane, ws.data_ptr(),
                                   (size_t)ws.numel(), current_stream()));
        variable_list out;
        for (int j = 0; j < r->k; ++j) {
            r->locations.push_back(piece(ints_, read + (int64_t)j * r->T, r->T));
            out.push_back(piece(gates, (int64_t)j * r->T, r->T));
        }
        if (r->want_loss) out.push_back(loss);
        // (as a variable: the gradient is that of these indices, and an index plane edited in place until then is refused.
        // The locations are not read again and are edited at will)
        r->read = piece(ints_, 0, read);
        ctx->save_for_backward({scores, r->read});
        ctx->saved_data["k"] = (int64_t)r->k;
        ctx->saved_data["normalize"] = r->normalize;
        return out;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor &scores = saved[0];
        const int32_t *i = ints(saved[1]);
        const c10::DeviceGuard guard(scores.device());
        const int k = (int)ctx->saved_data["k"].toInt(), T = (int)scores.size(0), E = (int)scores.size(1);
        std::vector<Tensor> gg(grads.begin(), grads.begin() + k);
        const Tensor dl = (int)grads.size() > k && grads[k].defined() ? grads[k].to(at::kFloat).contiguous() : Tensor();
        int64_t stride = T;
        bool any = dl.defined();
        for (Tensor &g : gg) {
            any |= g.defined();
            g = g.defined() ? g.contiguous() : at::zeros({T}, scores.options());
        }
        if (!any) return {Tensor(), Tensor()};
        if (spacing(gg) != T && k > 1) gg = {at::stack(gg)};        // (the indices' planes are T apart)
        Tensor out = at::empty_like(scores);
        PM_CALL(planmoe_route_bwd(scores.data_ptr(), pm_dtype(scores.scalar_type()), i, gg[0].data_ptr(), stride, T, E, k,
                                  ctx->saved_data["normalize"].toBool(), dl.defined() ? floats(dl) : nullptr, dl.defined() ? i + (int64_t)k * T : nullptr,
                                  0, out.data_ptr(), current_stream()));
        return {out, Tensor()};
    }
};

// ((indices, locations, gates), capacity, loss or None); None: scores the kernels do not take as they are
using Critical = std::tuple<std::vector<Tensor>, std::vector<Tensor>, std::vector<Tensor>, int64_t, std::optional<Tensor>>;
std::optional<Critical> extract_critical(const Tensor &scores_, int64_t top_k, bool want_loss, double capacity_factor, bool normalize, int64_t alignment)
{
    if (!scores_.is_cuda() || scores_.dim() != 2 || !pm_dtype_ok(scores_.scalar_type()) || scores_.size(0) < 1 || scores_.size(1) < 1 || top_k < 1 ||
        !(capacity_factor > 0) || scores_.numel() >= ((int64_t)1 << 31))
        return std::nullopt;
    Routed r;
    r.T = (int)scores_.size(0);
    r.E = (int)scores_.size(1);
    r.k = (int)std::min<int64_t>(top_k, r.E);
    if ((int64_t)r.k * r.T >= ((int64_t)1 << 31)) return std::nullopt;
    r.normalize = normalize;
    r.want_loss = want_loss;
    const c10::DeviceGuard guard(scores_.device());
    const Tensor scores = scores_.contiguous();
    variable_list out = Route::apply(scores, &r);
    std::optional<Tensor> loss;
    if (want_loss) {
        loss = out.back().scalar_type() == scores.scalar_type() ? out.back() : out.back().to(scores.scalar_type());
        out.pop_back();
    }
    int capacity = 0;
    PM_CALL(planmoe_capacity(r.T, r.E, r.k, capacity_factor, (int)alignment, &capacity));
    // (views of what the node has saved: their in-place changes are its)
    std::vector<Tensor> indices;
    for (int j = 0; j < r.k; ++j) indices.push_back(r.read.narrow(0, (int64_t)j * r.T, r.T));
    return Critical(std::move(indices), std::move(r.locations), std::move(out), capacity, loss);
}

} // namespace

void def_routing(pybind11::module_ &m)
{
    using release = pybind11::call_guard<pybind11::gil_scoped_release>;
    m.def("extract_critical", &extract_critical, release(), "routing of scores with the gates' and the loss's gradients");
    m.def("encode", &move<true>, release(), "tokens [T, M] to slots [E, capacity, M]");
    m.def("decode", &move<false>, release(), "slots to tokens [T, M]");
}
