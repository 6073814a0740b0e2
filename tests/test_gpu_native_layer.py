"""The layer with its built-in experts as one node (csrc/ext/layer.cpp) against the layer's own steps
(overlap.NATIVE_LAYER = False) on the same parameters: same routing, same codec values, the products summed in
the same order over fewer rows.  What may differ: bf16 roundings where a sum runs in another order, and a lossy
codec's step where its input differs in the last bit; a token within rounding of a routing tie (the two gate
kernels sum in different orders) would differ as a whole, which the seeds here avoid."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(native, codec, dtype, T, M, H, E, k, cf, train):
    import planmoe_amd
    from planmoe_amd import overlap
    overlap.NATIVE_LAYER = native
    try:
        torch.manual_seed(7)
        layer = planmoe_amd.moe_layer({"type": "top", "k": k, "capacity_factor": cf, "fp32_gate": True}, M,
                                      experts={"type": "ffn", "count_per_node": E, "hidden_size_per_expert": H},
                                      compress_name=codec).to(DEV).to(dtype)
        g = torch.Generator().manual_seed(T)
        x = torch.randn(T, M, generator=g).to(dtype).to(DEV).requires_grad_(train)
        if not train:
            with torch.no_grad():
                y = layer(x)
            torch.cuda.synchronize()
            return {"y": y, "l_aux": y.l_aux}
        gy = torch.randn(T, M, generator=g).to(dtype).to(DEV)
        y = layer(x)
        torch.autograd.backward([y, y.l_aux], [gy, torch.full((), 0.5, device=DEV).to(y.l_aux.dtype)])
        torch.cuda.synchronize()
        out = {"y": y.detach(), "l_aux": y.l_aux.detach(), "dx": x.grad}
        out.update({n: p.grad for n, p in layer.named_parameters()})
        return out
    finally:
        overlap.NATIVE_LAYER = True


def _compare(a, b, rel):
    assert set(a) == set(b)
    for name in a:
        p, q = a[name].double(), b[name].double()
        assert p.shape == q.shape and a[name].dtype == b[name].dtype, name
        assert bool(torch.isfinite(p).all()), name
        assert float((p - q).norm()) <= rel * float(q.norm()) + 1e-30, (name, float((p - q).norm() / q.norm()))


# one token; fewer tokens than experts; ragged; capacity that drops tokens; more experts than the gate's fused
# accumulation takes; row lengths of one piece, below and above a wave's 64 pieces
@pytest.mark.parametrize("T,M,H,E,k,cf", [(1, 64, 72, 4, 2, 1.0), (5, 264, 136, 8, 2, 1.25), (333, 520, 264, 4, 1, 0.5),
                                          (700, 1032, 256, 16, 2, 1.0), (257, 8, 8, 4, 4, 1.0), (2049, 256, 512, 8, 2, 1.2)])
@pytest.mark.parametrize("codec,dtype", [("no", torch.bfloat16), ("int8", torch.bfloat16), ("no", torch.float32), ("int8", torch.float32),
                                         ("zfp", torch.float32), ("lz", torch.float32)])
def test_native_layer_equals_its_steps(codec, dtype, T, M, H, E, k, cf):
    print("case", codec, dtype, T, M, H, E, k, cf, flush=True)
    # a bf16 gradient goes through three products and roundings of 2^-9 each way; int8 steps are 1 / 255 of a row's
    # range and flip rarely, zfp's likewise; fp32 sums of up to 2049 terms: 2049 2^-24 at the worst
    rel = 1e-2 if dtype == torch.bfloat16 else 1e-3 if codec in ("int8", "zfp") else 2e-5
    args = (codec, dtype, T, M, H, E, k, cf)
    _compare(_run(True, *args, True), _run(False, *args, True), rel)
    _compare(_run(True, *args, False), _run(False, *args, False), rel)


def test_native_layer_leaves_hooks_and_frozen_parameters_to_autograd():
    """Hooks on the experts keep the layer on its steps; parameters that need no gradient get none; the input alone may
    need one."""
    import planmoe_amd
    from planmoe_amd import overlap
    torch.manual_seed(3)
    layer = planmoe_amd.moe_layer({"type": "top", "k": 2, "fp32_gate": True}, 64,
                                  experts={"type": "ffn", "count_per_node": 4, "hidden_size_per_expert": 64}).to(DEV).bfloat16()
    x = torch.randn(40, 64, device=DEV).bfloat16()
    seen = []
    handle = layer.experts.register_forward_hook(lambda *a: seen.append(1))
    y = layer(x)
    assert seen and overlap.native_call(layer, layer.gates[0], x, 1, 1, 4) is None
    handle.remove()
    z = layer(x)
    assert len(seen) == 1 and torch.allclose(y.float(), z.float(), rtol=2e-2, atol=1e-2)
    for p in layer.parameters():
        p.requires_grad_(False)
    x.requires_grad_(True)
    layer(x).float().sum().backward()
    torch.cuda.synchronize()
    assert x.grad is not None and all(p.grad is None for p in layer.parameters())


def test_native_layer_refuses_tangents_and_leaves_global_hooks_to_the_steps():
    import planmoe_amd
    torch.manual_seed(3)
    layer = planmoe_amd.moe_layer({"type": "top", "k": 2, "fp32_gate": True}, 64,
                                  experts={"type": "ffn", "count_per_node": 4, "hidden_size_per_expert": 64}).to(DEV).bfloat16()
    x = torch.randn(40, 64, device=DEV).bfloat16()
    import torch.autograd.forward_ad as fw
    with fw.dual_level(), torch.no_grad(), pytest.raises((RuntimeError, NotImplementedError)):
        layer(fw.make_dual(x, torch.ones_like(x)))
    seen = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: seen.append(m))
    try:
        layer(x)
    finally:
        handle.remove()
    torch.cuda.synchronize()
    assert layer.experts in seen


# the codec on rows in registers against compress, then combine from the codes: bit for bit.  Rows of one piece, of no whole
# number of waves' pieces, of the longest kind; rows of one value, with NaN, infinities, negative zeros; choices without a slot
@pytest.mark.parametrize("M", [8, 520, 4096])
@pytest.mark.parametrize("k", [1, 2, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_layer_combine_equals_compress_and_combine(M, k, dtype):
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    print("case", M, k, dtype, flush=True)
    T, E, cap = 37, 4, 12
    g = torch.Generator().manual_seed(M + k)
    rows = torch.randn(E * cap, M, generator=g)
    rows[3] = 0.25
    rows[7, M // 2] = float("nan")
    rows[9, 0] = float("inf")
    rows[11, ::2] = -0.0
    rows[13] *= 1e-30 if dtype != torch.float16 else 1e-6
    rows = rows.to(dtype).to(DEV)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)], 1).int().contiguous().to(DEV)
    loc = torch.randint(0, cap + 3, (k, T), generator=g, dtype=torch.int32).to(DEV)
    gates, grad = torch.rand(k, T, generator=g).to(DEV), torch.randn(T, M, generator=g).to(dtype).to(DEV)
    out = torch.empty(T, M, dtype=dtype, device=DEV)
    check(lib.planmoe_layer_combine(ops._ptr(rows), ops._dt(rows, "t"), 1, ops._ptr(gates), ops._ptr(idx), ops._ptr(loc), T, k, T, M, E, cap,
                                    ops._ptr(out), ops._stream(rows)))
    codes, bias, scale = ops.int8_compress(rows)
    want = ops.combine_int8(codes, bias, scale, list(idx), list(loc), list(gates), T, cap)
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    same = (out.view(bits) == want.view(bits)) | (out.isnan() & want.isnan())
    torch.cuda.synchronize()
    assert bool(same.all())
    # the backward pass: gate gradients, and rows by their slots (unique slots only: two tokens on one slot would race)
    if k == 1:
        loc, idx = (torch.arange(T) // E).int()[None].contiguous().to(DEV), (torch.arange(T) % E).int()[None].contiguous().to(DEV)
        grad_rows, gg = torch.zeros_like(rows), torch.empty(k, T, device=DEV)
        check(lib.planmoe_layer_combine_bwd(ops._ptr(grad), ops._ptr(rows), ops._dt(rows, "t"), 1, ops._ptr(gates), ops._ptr(idx), ops._ptr(loc), T, k, T, M,
                                            E, cap, ops._ptr(grad_rows), ops._ptr(gg), ops._stream(rows)))
        seen = ops.int8_decompress(codes, bias, scale)
        slot = (idx[0] * cap + loc[0]).long()
        gated = (gates[0][:, None] * grad.float()).to(dtype)
        c2 = ops.int8_compress(gated)
        wanted = ops.int8_decompress(*c2)
        dots, mag = (seen[slot].double() * grad.double()).sum(1), (seen[slot].double() * grad.double()).abs().sum(1)
        torch.cuda.synchronize()
        assert torch.equal(grad_rows[slot].view(bits), wanted.view(bits))
        fine = torch.isfinite(dots)
        assert bool(((gg[0].double() - dots).abs() <= (M + 2) * 2.0 ** -24 * mag + 1e-30)[fine].all())


def _layer(dtype, codec="no", M=64, H=72, E=4, k=2, cf=1.25, cls=None):
    import planmoe_amd
    torch.manual_seed(3)
    return (cls or planmoe_amd.moe_layer)({"type": "top", "k": k, "capacity_factor": cf, "fp32_gate": True}, M,
                                          experts={"type": "ffn", "count_per_node": E, "hidden_size_per_expert": H},
                                          compress_name=codec).to(DEV).to(dtype)


def test_replaced_methods_are_called(monkeypatch):
    """The forward of the experts replaced on the object or in the class, expert_local overridden or replaced: the layer goes
    through them."""
    from planmoe_amd.experts import FusedExpertsNetwork
    from planmoe_amd.moe_layer import MOELayer
    x = torch.randn(40, 64, device=DEV).bfloat16()
    seen = []

    def twice(inner):
        def call(*args):
            seen.append(1)
            return inner(*args) * 2
        return call

    with torch.no_grad():
        plain = _layer(torch.bfloat16)(x)
        layer = _layer(torch.bfloat16)
        layer.experts.forward = twice(layer.experts.forward)
        got = [layer(x)]
        layer = _layer(torch.bfloat16)
        layer.expert_local = twice(layer.expert_local)
        got.append(layer(x))

        class Mine(MOELayer):
            def expert_local(self, *args):
                return twice(super().expert_local)(*args)

        got.append(_layer(torch.bfloat16, cls=Mine)(x))
        layer = _layer(torch.bfloat16)
        for cls, name in ((FusedExpertsNetwork, "forward"), (MOELayer, "expert_local")):
            with monkeypatch.context() as m:
                m.setattr(cls, name, twice(getattr(cls, name)))
                got.append(layer(x))
    torch.cuda.synchronize()
    assert len(seen) == 5
    for y in got:                                # (the products of the steps sum in another order: bf16 roundings)
        assert float((y.double() - 2 * plain.double()).norm()) <= 1e-2 * float(2 * plain.double().norm())


def _pass(layer, x, gy):
    layer.zero_grad()
    x = x.clone().requires_grad_(True)
    y = layer(x)
    y.backward(gy)
    torch.cuda.synchronize()
    return {"y": y.detach(), "dx": x.grad, **{n: p.grad for n, p in layer.named_parameters()}}


@pytest.mark.parametrize("codec,dtype", [("no", torch.bfloat16), ("no", torch.float32), ("int8", torch.bfloat16), ("int8", torch.float32),
                                         ("zfp", torch.float32), ("lz", torch.float32)])
def test_gradient_that_is_not_aligned(codec, dtype):
    """What torch.cat sends back to a part of its result is contiguous and begins anywhere."""
    layer = _layer(dtype, codec)
    x, gy = torch.randn(40, 64, device=DEV).to(dtype), torch.randn(40, 64, device=DEV).to(dtype)
    off = torch.cat([gy.new_zeros(1), gy.flatten()])[1:].view_as(gy)
    assert off.is_contiguous() and off.data_ptr() % 16 != 0
    want, got = _pass(layer, x, gy), _pass(layer, x, off)
    for name in want:
        assert torch.equal(want[name], got[name]), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_weights_that_are_not_aligned(dtype):
    """Parameters that are views of a flat buffer, biases that are columns of one."""
    layer = _layer(dtype)
    x, gy = torch.randn(40, 64, device=DEV).to(dtype), torch.randn(40, 64, device=DEV).to(dtype)
    want = _pass(layer, x, gy)
    experts = layer.experts
    flat = torch.cat([torch.zeros(1, dtype=dtype, device=DEV)] + [p.detach().flatten() for p in experts.parameters()])
    at = 1
    for name, p in list(experts.named_parameters()):
        view = flat[at:at + p.numel()].view(p.shape)
        assert view.data_ptr() % 16 != 0
        setattr(experts, name, torch.nn.Parameter(view))
        at += p.numel()
    # (the products now run over whole buffers: bf16 roundings, and sums of up to 72 terms in another order)
    _compare(_pass(layer, x, gy), want, 1e-2 if dtype == torch.bfloat16 else 2e-5)
    # the experts alone, with rows and a gradient that are not aligned either, a bias with gaps between its values
    rows = torch.randn(1 + 4 * 20 * 64, device=DEV).to(dtype)[1:].view(4, 20, 64)
    whole = experts(rows.clone(), layer).detach()
    experts.batched_fc1_bias = torch.nn.Parameter(experts.batched_fc1_bias.detach()[..., None].repeat(1, 1, 3)[..., 1])
    got = []
    for off in (True, False):
        r = (rows if off else rows.clone()).detach().requires_grad_(True)
        g = rows if off else rows.clone()
        layer.zero_grad()
        y = experts(r, layer)
        y.backward(g)
        got.append([y.detach(), r.grad] + [p.grad for p in experts.parameters()])
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], whole)
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_fp32_layer_with_two_million_slots_an_expert():
    """The number of slots is no row length: it has no bound but the slots' numbers (int32)."""
    T, cf = 8, 524290.0                          # capacity 4 cf: 2097160, 2 GiB over 256 rows of 4-byte values and 8
    args = ("no", torch.float32, T, 8, 8, 2, 1, cf, True)
    _compare(_run(True, *args), _run(False, *args), 2e-5)


# the codes kept for the backward pass: what the codec gives for the rows that hold a token, and nothing else written; the
# output, the gradients of the gates and of the rows are the same bits as with the rows themselves
@pytest.mark.parametrize("M", [8, 520, 4096])
@pytest.mark.parametrize("k", [1, 2, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_layer_combine_from_kept_codes(M, k, dtype):
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    print("case", M, k, dtype, flush=True)
    T, E, cap = 37, 4, 29
    g = torch.Generator().manual_seed(M + k)
    rows = torch.randn(E * cap, M, generator=g)
    rows[3] = 0.25
    rows[7, M // 2] = float("nan")
    rows[9, 0] = float("inf")
    rows[11, ::2] = -0.0
    rows[13] *= 1e-30 if dtype != torch.float16 else 1e-6
    rows = rows.to(dtype).to(DEV)
    # pair n of a token and a choice has slot n % (cap + 3) of expert n / (cap + 3): every slot once, some behind the capacity
    n = torch.arange(T * k).view(T, k).t()
    idx, loc = (n // (cap + 3)).int().contiguous().to(DEV), (n % (cap + 3)).int().contiguous().to(DEV)
    gates, grad = torch.rand(k, T, generator=g).to(DEV), torch.randn(T, M, generator=g).to(dtype).to(DEV)
    out, want = (torch.empty(T, M, dtype=dtype, device=DEV) for _ in range(2))
    codes = torch.full((E * cap, M), 77, dtype=torch.uint8, device=DEV)
    bias, scale = (torch.full((E * cap,), 5.0, dtype=dtype, device=DEV) for _ in range(2))
    planes = (ops._ptr(gates), ops._ptr(idx), ops._ptr(loc), T, k, T, M, E, cap)
    check(lib.planmoe_layer_combine(ops._ptr(rows), ops._dt(rows, "t"), 1, *planes, ops._ptr(want), ops._stream(rows)))
    check(lib.planmoe_layer_combine_keep(ops._ptr(rows), ops._dt(rows, "t"), *planes, ops._ptr(out), ops._ptr(codes), ops._ptr(bias),
                                         ops._ptr(scale), ops._stream(rows)))
    all_codes, all_bias, all_scale = ops.int8_compress(rows)
    grad_rows, wanted_rows = torch.full_like(rows, 7.0), torch.full_like(rows, 7.0)
    gg, wanted_gates = torch.empty(k, T, device=DEV), torch.empty(k, T, device=DEV)
    check(lib.planmoe_layer_combine_bwd(ops._ptr(grad), ops._ptr(rows), ops._dt(rows, "t"), 1, *planes, ops._ptr(wanted_rows), ops._ptr(wanted_gates),
                                        ops._stream(rows)))
    check(lib.planmoe_layer_combine_bwd_codes(ops._ptr(grad), ops._ptr(codes), ops._ptr(bias), ops._ptr(scale), ops._dt(rows, "t"), *planes,
                                              ops._ptr(grad_rows), ops._ptr(gg), ops._stream(rows)))
    torch.cuda.synchronize()
    live = loc < cap
    used = torch.zeros(E * cap, dtype=torch.bool, device=DEV)
    used[(idx * cap + loc).long()[live]] = True
    assert int(used.sum()) == int(live.sum()) and int((~live).sum()) > 0

    def same(a, b):
        bits = torch.int32 if dtype == torch.float32 else torch.int16
        return bool(((a.view(bits) == b.view(bits)) | (a.isnan() & b.isnan())).all())
    assert torch.equal(codes[used], all_codes.view(E * cap, M)[used]) and bool((codes[~used] == 77).all())
    assert same(bias[used], all_bias.view(-1)[used]) and same(scale[used], all_scale.view(-1)[used])
    assert bool((bias[~used] == 5.0).all()) and bool((scale[~used] == 5.0).all())
    assert same(out, want) and same(grad_rows, wanted_rows)
    assert bool(((gg == wanted_gates) | (gg.isnan() & wanted_gates.isnan())).all())


def test_int8_training_holds_no_more_than_its_steps():
    """Between the passes the second product's output is held as codes, a byte a value, as the steps hold it."""
    from planmoe_amd import overlap

    def held(native, dtype):
        overlap.NATIVE_LAYER = native
        kept = {}

        def pack(t):
            kept[t.untyped_storage().data_ptr()] = t.untyped_storage().nbytes()
            return t
        try:
            layer, x = _layer(dtype, "int8", M=256, H=64), torch.randn(512, 256, device=DEV).to(dtype).requires_grad_(True)
            with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
                y = layer(x)
            y.float().sum().backward()
            torch.cuda.synchronize()
        finally:
            overlap.NATIVE_LAYER = True
        return sum(kept.values())

    for dtype in (torch.bfloat16, torch.float32):
        native, steps = held(True, dtype), held(False, dtype)
        print("held", dtype, native, steps, flush=True)
        assert native <= steps + 4096            # (a plane or a scalar that the steps take apart)


@pytest.mark.parametrize("codec,dtype", [("no", torch.bfloat16), ("int8", torch.bfloat16), ("no", torch.float32), ("zfp", torch.float32),
                                         ("lz", torch.float32)])
def test_native_layer_on_a_stream_of_its_own(codec, dtype):
    """The forward pass on another stream, behind work that is still running there; the backward pass asked for from the
    stream that was current before: everything is launched, and its memory used, on the forward pass's stream."""
    layer = _layer(dtype, codec)
    g = torch.Generator(device=DEV).manual_seed(1)
    x, gy = (torch.randn(300, 64, device=DEV, generator=g).to(dtype) for _ in range(2))
    want = _pass(layer, x, gy)
    layer.zero_grad()
    v, stream = torch.zeros_like(x).requires_grad_(True), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        torch.cuda._sleep(20_000_000)            # (about 10 ms: what does not wait for the copy below sees other values)
        with torch.no_grad():
            v.copy_(x)
        y = layer(v)
    y.backward(gy)
    torch.cuda.current_stream().wait_stream(stream)
    got = {"y": y.detach(), "dx": v.grad, **{n: p.grad for n, p in layer.named_parameters()}}
    torch.cuda.synchronize()
    for name in want:
        assert torch.equal(want[name], got[name]), name


# the zfp codec as it reaches the layer's rows against the coder and the decoder, bit for bit: fields that spend their bits on few
# planes and on many, whose budget ends in and between planes and that never reach it, zeros, subnormals, infinities, NaN, the largest values
@pytest.mark.parametrize("M", [4, 64, 1028])
def test_layer_zfp_rows_equal_compress_and_decompress(M):
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    print("case", M, flush=True)
    E, cap = 8, 64
    g = torch.Generator().manual_seed(M)
    rows = torch.randn(E, cap, M, generator=g)
    at = torch.arange(M) / M
    rows[1] = torch.sin(at * torch.randint(1, 9, (cap, 1), generator=g)) + 1e-3 * rows[1]
    rows[2] = torch.exp(20 * rows[2])                                                         # a few values tell
    rows[3] *= torch.rand(cap, M, generator=g) < 0.1
    rows[4] = rows[4].sign() * 2.0 ** torch.randint(-149, 128, (cap, M), generator=g).float()
    rows[5, :16], rows[5, 16:32], rows[5, 32:48] = 0.75, torch.randint(-4, 5, (16, M), generator=g).float(), rows[5, 32:48] * 1e-42
    rows[5, 48:52], rows[5, 52:56], rows[5, 56:] = 0.0, 3.4e38, rows[5, 56:] * 2.0 ** -126
    special = torch.tensor([float("inf"), float("-inf"), float("nan"), -0.0, 1.0, 3e38, 1e-40])
    rows[6] = torch.where(torch.rand(cap, M, generator=g) < 0.05, special[torch.randint(0, 7, (cap, M), generator=g)], rows[6])
    rows[7] = special[torch.randint(0, 7, (cap, M), generator=g)]
    counts = torch.tensor([[64, 30, 64, 61, 40, 64, 0, 63], [0, 5, 70, 2, 24, 0, 64, 0]], dtype=torch.int32)
    rows, counts = rows.to(DEV), counts.to(DEV)
    stream = ops.zfp_compress(rows.view(E * cap, M), M, E * cap, 2)
    want = ops.zfp_decompress(stream, M, E * cap, 2).view(E, cap, M)
    for keep in (False, True):
        got, kept = rows.clone(), torch.zeros_like(stream)
        check(lib.planmoe_layer_zfp_rows(ops._ptr(got), M, E, cap, ops._ptr(counts), 2, ops._ptr(kept) if keep else None,
                                         kept.numel() * kept.element_size() if keep else 0, ops._stream(got)))
        torch.cuda.synchronize()
        for e, n in enumerate(counts.sum(0).clamp(max=cap).tolist()):
            n = (n + 3) // 4 * 4
            assert torch.equal(got[e, :n].view(torch.int32), want[e, :n].view(torch.int32)), (e, keep)
            assert torch.equal(got[e, n:].view(torch.int32), rows[e, n:].view(torch.int32)), (e, keep)
            if keep:
                size = cap * M                   # (a byte a value)
                a, b = (t.view(torch.uint8)[e * size:e * size + n * M] for t in (kept, stream))
                assert torch.equal(a, b) and not kept.view(torch.uint8)[e * size + n * M:(e + 1) * size].any(), e


@pytest.mark.parametrize("T,M,E,k,cap", [(1, 4, 4, 1, 4), (333, 520, 4, 2, 100), (100, 1028, 8, 3, 64), (257, 64, 16, 2, 8)])
def test_layer_zfp_dispatch_and_combine_backward_equal_the_steps(T, M, E, k, cap):
    """Against planmoe_dispatch_zfp, planmoe_zfp_decompress and planmoe_bwd_gate_zfp, bit for bit; tokens that take no slot."""
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    print("case", T, M, E, k, cap, flush=True)
    g = torch.Generator(device=DEV).manual_seed(T + M)
    x, grad = torch.randn(T, M, generator=g, device=DEV), torch.randn(T, M, generator=g, device=DEV)
    routed = ops.route_topk(torch.softmax(torch.randn(T, E, generator=g, device=DEV), 1), k)
    idx, loc = (torch.stack(list(routed[n])).int().contiguous() for n in ("indices", "locations"))
    gates = torch.rand(k, T, generator=g, device=DEV)
    counts = torch.stack([torch.bincount(i.long(), minlength=E) for i in idx]).int().contiguous()
    ws = torch.empty(lib.planmoe_layer_zfp_workspace_bytes(E, cap), dtype=torch.uint8, device=DEV).fill_(0x7f)      # (no slot of before helps)
    rows, grad_rows = torch.full((E, cap, M), 7.0, device=DEV), torch.full((E, cap, M), 7.0, device=DEV)
    grad_gates = torch.full((k, T), 7.0, device=DEV)
    check(lib.planmoe_layer_zfp_dispatch(ops._ptr(x), ops._ptr(idx), ops._ptr(loc), T, k, T, M, E, cap, ops._ptr(counts), ops._ptr(rows),
                                         ops._ptr(ws), ws.numel(), ops._stream(x)))
    want = ops.zfp_decompress(ops.dispatch_zfp(x, list(idx), list(loc), None, E, cap), M, E * cap, 2).view(E, cap, M)
    seen = ops.zfp_compress(torch.randn(E * cap, M, generator=g, device=DEV), M, E * cap, 2)
    ws.fill_(0x7f)
    check(lib.planmoe_layer_zfp_combine_bwd(ops._ptr(seen), ops._ptr(grad), ops._ptr(gates), ops._ptr(idx), ops._ptr(loc), T, k, T, M, E, cap,
                                            ops._ptr(counts), ops._ptr(grad_rows), ops._ptr(grad_gates), ops._ptr(ws), ws.numel(), ops._stream(x)))
    want_rows = ops.zfp_decompress(ops.dispatch_zfp(grad, list(idx), list(loc), list(gates), E, cap), M, E * cap, 2).view(E, cap, M)
    want_gates = ops.bwd_gate_zfp(seen, grad, list(idx), list(loc), E, cap)
    torch.cuda.synchronize()
    assert torch.equal(grad_gates, want_gates.view(k, T))
    for e, n in enumerate(counts.sum(0).clamp(max=cap).tolist()):
        n = (n + 3) // 4 * 4
        assert torch.equal(rows[e, :n], want[e, :n]) and bool((rows[e, n:] == 7.0).all()), e
        assert torch.equal(grad_rows[e, :n], want_rows[e, :n]) and bool((grad_rows[e, n:] == 7.0).all()), e


# up to 32 tokens and 16 experts the gate, the routing and the rows are one launch (33 tokens, 17 experts: two): the same bits as the
# chain of two launches.  Work-groups of four tokens, rows of one vector and of no whole number of a wave's, capacities that drop choices
@pytest.mark.parametrize("T,M,E,k,cap", [(1, 8, 1, 1, 4), (3, 64, 4, 2, 4), (4, 1032, 8, 4, 2), (5, 520, 9, 3, 4), (31, 256, 16, 2, 4),
                                         (32, 2048, 8, 2, 12), (32, 64, 2, 2, 8), (33, 256, 16, 2, 4), (8, 64, 17, 1, 4)])
@pytest.mark.parametrize("codec", [0, 1])
@pytest.mark.parametrize("dtype,fp32_gate", [(torch.bfloat16, True), (torch.bfloat16, False), (torch.float32, True), (torch.float16, True)])
def test_layer_dispatch_of_few_tokens_equals_two_launches(T, M, E, k, cap, codec, dtype, fp32_gate):
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    print("case", T, M, E, k, cap, codec, dtype, fp32_gate, flush=True)
    g = torch.Generator().manual_seed(T + M + E)
    x, wg = torch.randn(T, M, generator=g).to(dtype).to(DEV), (torch.randn(E, M, generator=g) * M ** -0.5).to(dtype).to(DEV)
    x[T // 2] = 0.5                              # (a row of one value: no scale)
    x[0, 0] = -0.0
    kw = dict(fp32_gate=fp32_gate, want_scores=True, want_counts=True)
    if codec:
        want = ops.forward_int8(x, wg, k, cap, **kw)
        want["rows"] = ops.int8_decompress(want["codes"], want["bias"], want["scale"])
    else:
        want = ops.forward_plain(x, wg, k, cap, **kw)
        want["rows"] = want["dispatched"]
    score = torch.float32 if fp32_gate else dtype
    idx, loc, counts = (torch.full(s, -7, dtype=torch.int32, device=DEV) for s in ((k, T), (k, T), (k, E)))
    gates, scores = torch.full((k, T), 7.0, dtype=score, device=DEV), torch.full((T, E), 7.0, dtype=score, device=DEV)
    l_aux, rows = torch.full((), 7.0, device=DEV), torch.full((E * cap, M), 7.0, dtype=dtype, device=DEV)
    ws = torch.empty(lib.planmoe_forward_workspace_bytes(T, E, k), dtype=torch.uint8, device=DEV).fill_(0x7f)
    check(lib.planmoe_layer_dispatch(ops._ptr(x), ops._ptr(wg), ops._dt(x, "t"), int(fp32_gate), None, T, M, E, k, 1, cap, codec, ops._ptr(idx),
                                     ops._ptr(loc), ops._ptr(gates), T, ops._ptr(scores), ops._ptr(l_aux), ops._ptr(counts), ops._ptr(rows),
                                     ops._ptr(ws), ws.numel(), ops._stream(x)))
    alone = ops.gate_route(x, wg, k, **kw)
    torch.cuda.synchronize()
    for name, got in (("indices", idx), ("locations", loc), ("gates", gates), ("scores", scores), ("counts", counts), ("l_aux", l_aux)):
        assert torch.equal(got, want[name].view(got.shape)), name
        assert torch.equal(alone[name].view(got.shape), got), name
    used = torch.zeros(E * cap, dtype=torch.bool, device=DEV)
    used[(idx.long() * cap + loc)[loc < cap]] = True
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    assert torch.equal(rows[used].view(bits), want["rows"].view(E * cap, M)[used].view(bits)) and bool((rows[~used] == 7.0).all())


# (a routing group of 16 tokens, full and one short of it)
@pytest.mark.parametrize("T,M,E,k,cap", [(15, 264, 16, 2, 4), (16, 2056, 8, 2, 4), (16, 64, 3, 3, 16)])
@pytest.mark.parametrize("codec", [0, 1])
@pytest.mark.parametrize("dtype,fp32_gate", [(torch.bfloat16, True), (torch.float32, True)])
def test_layer_dispatch_of_sixteen_tokens_equals_two_launches(T, M, E, k, cap, codec, dtype, fp32_gate):
    test_layer_dispatch_of_few_tokens_equals_two_launches(T, M, E, k, cap, codec, dtype, fp32_gate)


# The first product of up to 32 tokens routes them itself: the bits of the dispatch and the product behind it.  Columns of a work-group 32,
# 64 and 128, read past the caches and not; rows that are no whole steps of the reduction; capacities that drop choices, 16 rows and (two
# launches) 20; 16 experts, 17 and 33 tokens (two launches); experts without a row
@pytest.mark.parametrize("T,M,E,k,cap,H", [(1, 8, 1, 1, 4, 8), (3, 64, 4, 2, 4, 200), (5, 1032, 9, 3, 4, 520), (31, 256, 16, 2, 4, 1024), (32, 2048, 8, 2, 12, 136),
                                           (20, 2056, 4, 2, 16, 1032), (20, 4096, 4, 2, 16, 1032), (8, 1024, 8, 2, 4, 4096), (17, 520, 16, 4, 8, 2040), (32, 264, 8, 2, 16, 4088),
                                           (30, 64, 2, 2, 20, 64), (33, 256, 16, 2, 8, 264), (8, 64, 17, 1, 4, 64), (4, 4096, 8, 4, 2, 3000)])
@pytest.mark.parametrize("codec", [0, 1])
@pytest.mark.parametrize("skewed", [False, True])
def test_first_product_that_routes_equals_dispatch_and_product(T, M, E, k, cap, H, codec, skewed):
    _first_product(T, M, E, k, cap, H, codec, skewed)


def _first_product(T, M, E, k, cap, H, codec, skewed, with_bias=True, normalize=1, gap=0, dtype=torch.bfloat16, fp32_gate=True):
    """gap: entries of a plane behind its tokens."""
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    print("case", T, M, E, k, cap, H, codec, skewed, with_bias, normalize, gap, dtype, fp32_gate, flush=True)
    g = torch.Generator(device=DEV).manual_seed(T + M + E)
    randn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, wg, w1 = randn(T, M).to(dtype), (randn(E, M) * M ** -0.5).to(dtype), (randn(E, M, H) * M ** -0.5).to(dtype)
    b1 = randn(E, H).to(dtype) if with_bias else None
    if skewed:                                   # everything to the last experts, and values that are not finite
        wg[:] = torch.arange(E, device=DEV)[:, None] / M
        x = x.abs()
        x[T // 2, 1] = float("nan")
        x[T - 1, 0] = float("inf")
    else:
        x[T // 2] = 0.5                          # (a row of one value: no scale)
        x[0, 0] = -0.0
    hint, stride = min(cap, (T * k + E - 1) // E), T + gap
    ws = torch.empty(lib.planmoe_forward_workspace_bytes(T, E, k), dtype=torch.uint8, device=DEV)

    def outputs():
        ints = [torch.full(s, -7, dtype=torch.int32, device=DEV) for s in ((k, stride), (k, stride), (k, E))]
        floats = [torch.full((k, stride), 7.0, dtype=torch.float32 if fp32_gate else dtype, device=DEV), torch.full((), 7.0, device=DEV)]
        return ints, floats, torch.full((E, cap, M), 7.0, dtype=dtype, device=DEV), torch.full((E, cap, H), 7.0, dtype=dtype, device=DEV)

    ints, floats, rows, h = outputs()
    check(lib.planmoe_layer_dispatch_product(ops._ptr(x), ops._ptr(wg), ops._dt(x, "t"), int(fp32_gate), T, M, E, k, normalize, cap, codec, ops._ptr(ints[0]),
                                             ops._ptr(ints[1]), ops._ptr(floats[0]), stride, ops._ptr(floats[1]), ops._ptr(ints[2]), ops._ptr(w1), ops._ptr(b1), H,
                                             hint, ops._ptr(rows), ops._ptr(h), ops._ptr(ws), ws.numel(), ops._stream(x)))
    want_ints, want_floats, want_rows, want_h = outputs()
    check(lib.planmoe_layer_dispatch(ops._ptr(x), ops._ptr(wg), ops._dt(x, "t"), int(fp32_gate), None, T, M, E, k, normalize, cap, codec, ops._ptr(want_ints[0]),
                                     ops._ptr(want_ints[1]), ops._ptr(want_floats[0]), stride, None, ops._ptr(want_floats[1]), ops._ptr(want_ints[2]),
                                     ops._ptr(want_rows), ops._ptr(ws), ws.numel(), ops._stream(x)))
    ops.expert_gemm("nn", want_rows, w1, b1, relu=True, live=want_ints[2], rows_hint=hint, out=want_h)
    torch.cuda.synchronize()
    # (then the rows stay where they are; a product in 32 or 64 columns has them where that is no more work-groups than there are compute units)
    units = torch.cuda.get_device_properties(0).multi_processor_count
    one = T <= 32 and E <= 16 and cap <= 16 and k <= 4 and dtype == torch.bfloat16 and fp32_gate and (H + 127) // 128 * E <= units
    assert bool((rows == 7.0).all()) == one
    bits = lambda t: t.view(torch.int32 if t.dtype == torch.float32 else torch.int16)
    for got, want in zip(ints, want_ints):
        assert torch.equal(got, want)
    for got, want in zip(floats + [h], want_floats + [want_h]):
        assert torch.equal(bits(got), bits(want))


# the same: gates as they are, no bias, planes wider than the tokens; and what has two launches: more work-groups than there are compute units (and as
# many), five choices, a gate in bf16, rows in fp32
@pytest.mark.parametrize("T,M,E,k,cap,H,kw", [
    (9, 520, 8, 2, 8, 264, dict(with_bias=False)), (32, 1024, 16, 3, 8, 72, dict(normalize=0)), (7, 264, 4, 2, 8, 2056, dict(gap=25)),
    (20, 2048, 8, 4, 16, 520, dict(with_bias=False, normalize=0, gap=1)), (8, 64, 16, 2, 4, 2048, {}), (8, 64, 16, 2, 4, 2056, {}), (8, 64, 8, 5, 8, 136, {}),
    (8, 264, 8, 2, 8, 136, dict(fp32_gate=False)), (8, 264, 8, 2, 8, 136, dict(dtype=torch.float32, gap=3)), (16, 128, 4, 4, 16, 4096, dict(gap=7, normalize=0))])
@pytest.mark.parametrize("codec", [0, 1])
def test_first_product_that_routes_with_other_options(T, M, E, k, cap, H, kw, codec):
    _first_product(T, M, E, k, cap, H, codec, False, **kw)


# without autograd a pass lies in one buffer: the same bits as the pass that a backward pass may follow, gates in 16 bits among them
@pytest.mark.parametrize("codec,dtype,fp32_gate", [("no", torch.bfloat16, True), ("no", torch.bfloat16, False), ("int8", torch.bfloat16, False),
                                                   ("int8", torch.float32, True), ("zfp", torch.float32, True), ("no", torch.float32, False)])
@pytest.mark.parametrize("T,k", [(1, 1), (19, 2), (300, 3)])
def test_inference_equals_the_pass_with_autograd(codec, dtype, fp32_gate, T, k):
    import planmoe_amd
    torch.manual_seed(T)
    layer = planmoe_amd.moe_layer({"type": "top", "k": k, "capacity_factor": 1.1, "fp32_gate": fp32_gate}, 136,
                                  experts={"type": "ffn", "count_per_node": 4, "hidden_size_per_expert": 200}, compress_name=codec).to(DEV).to(dtype)
    x = torch.randn(T, 136, device=DEV).to(dtype)
    want = layer(x)
    with torch.no_grad():
        got = [layer(x) for _ in range(2)]
    torch.cuda.synchronize()
    assert want.requires_grad
    for y in got:
        assert torch.equal(y, want) and torch.equal(y.l_aux, want.l_aux) and y.l_aux.dtype == want.l_aux.dtype


# Everything asked for (the reductions share their launches, the gate's part is added in the combine) against one gradient at a time
# (each by its own launches): the same sums in the same order.  Up to 8 experts and rows of at most 8 KB: dx in one pass; 9 and 16
# experts: two groups of eight in the gate weight's gradient; M 4104 and, in fp32, 2056: rows above 8 KB; 4099 tokens: two a wave, one left.
@pytest.mark.parametrize("T,M,H,E,k,cf", [(4, 8, 8, 1, 1, 1.0), (5, 264, 136, 8, 2, 1.25), (333, 1024, 264, 4, 1, 0.5), (700, 2056, 256, 3, 2, 1.0),
                                          (40, 4104, 16, 4, 2, 1.0), (4099, 64, 72, 8, 2, 1.0), (130, 520, 72, 9, 3, 1.0), (2049, 256, 512, 16, 2, 1.2)])
@pytest.mark.parametrize("codec,dtype,fp32_gate", [("no", torch.bfloat16, True), ("no", torch.bfloat16, False), ("int8", torch.bfloat16, True),
                                                   ("no", torch.float32, True), ("int8", torch.float32, True), ("zfp", torch.float32, True)])
@pytest.mark.parametrize("with_loss", [True, False])
def test_all_gradients_equal_one_at_a_time(codec, dtype, fp32_gate, T, M, H, E, k, cf, with_loss):
    import planmoe_amd
    E = (E + 3) // 4 * 4 if codec == "zfp" else E          # (its extents are multiples of four)
    M = min(M, 4096) if dtype == torch.float32 else M            # (as far as the node goes)
    print("case", codec, dtype, fp32_gate, T, M, H, E, k, cf, with_loss, flush=True)
    torch.manual_seed(T)
    layer = planmoe_amd.moe_layer({"type": "top", "k": k, "capacity_factor": cf, "fp32_gate": fp32_gate}, M,
                                  experts={"type": "ffn", "count_per_node": E, "hidden_size_per_expert": H}, compress_name=codec).to(DEV).to(dtype)
    x = torch.randn(T, M, device=DEV).to(dtype).requires_grad_(True)
    gy = torch.randn(T, M, device=DEV).to(dtype)
    params = [x] + list(layer.parameters())

    def grads(wanted):
        for p in params: p.requires_grad_(any(p is w for w in wanted))
        y = layer(x)
        out = [y, y.l_aux] if with_loss else [y]
        got = torch.autograd.grad(out, wanted, [gy, torch.full_like(y.l_aux, 0.5)] if with_loss else [gy], allow_unused=True)
        torch.cuda.synchronize()
        return got

    whole = grads(params)
    for p, got in zip(params, whole):
        one = grads([p])[0]
        assert got is not None and torch.equal(got, one), (tuple(p.shape), float((got.double() - one.double()).abs().max()))


# fp32, products in three bf16 parts a value among them: the node's, over the rows in use, have the bits of the steps', over the whole buffer.  Capacities
# on either side of the rows that are left to the fp32 matrix cores, some beyond the rows expected
@pytest.mark.parametrize("codec,cf", [("no", 1.0), ("no", 1.25), ("no", 1.5), ("lz", 1.25)])
@pytest.mark.parametrize("T", [240, 1000, 3000])
def test_native_layer_has_the_bits_of_its_steps_in_fp32(codec, cf, T):
    args = (codec, torch.float32, T, 512, 1024, 8, 2, cf)
    for train in (False, True):
        got, want = _run(True, *args, train), _run(False, *args, train)
        for name in ["y", "l_aux"] + (["experts.batched_fc1_w", "experts.batched_fc2_w"] if train else []):      # (other sums have kernels of their own)
            assert torch.equal(got[name], want[name]), (name, train)


# the same in fp32 where products go over in three bf16 parts a value (more than 64 rows an expert, rows of 256 values and more): the product
# under the relu keeps one order of sums in both passes, so a frozen copy, an evaluation and a checkpoint's first run see the same bits
@pytest.mark.parametrize("codec", ["no", "int8", "zfp", "lz"])
@pytest.mark.parametrize("T", [500, 4096])
def test_inference_equals_the_pass_with_autograd_in_larger_fp32_products(codec, T):
    layer = _layer(torch.float32, codec, M=512, H=1024, E=8)
    x = torch.randn(T, 512, device=DEV, generator=torch.Generator(device=DEV).manual_seed(T))
    want = layer(x)
    with torch.no_grad():
        got = layer(x)
    torch.cuda.synchronize()
    assert want.requires_grad and torch.equal(got, want) and torch.equal(got.l_aux, want.l_aux)


def test_reentrant_checkpoint_gives_the_gradients_of_the_plain_pass_in_fp32():
    """Its first run is without autograd, its second with it."""
    from torch.utils.checkpoint import checkpoint
    layer = _layer(torch.float32, M=512, H=1024, E=8)
    g = torch.Generator(device=DEV).manual_seed(1)
    x, gy = (torch.randn(4096, 512, device=DEV, generator=g) for _ in range(2))
    want = _pass(layer, x, gy)
    layer.zero_grad()
    v = x.clone().requires_grad_(True)
    y = checkpoint(layer, v, use_reentrant=True)
    y.backward(gy)
    got = {"y": y.detach(), "dx": v.grad, **{n: p.grad for n, p in layer.named_parameters()}}
    torch.cuda.synchronize()
    for name in want:
        assert torch.equal(want[name], got[name]), name


def test_native_layer_equals_its_steps_in_the_largest_parts():
    """fp32 rows that are a tile of 256 x 128 in three parts a value, with the codec whose steps show a last bit."""
    from planmoe_amd import ops
    assert ops.expert_gemm_kernel("nt", torch.float32, 16, 512, 1024, 1024, counted=True, rows_hint=512) == "f32 parts 256x128"
    args = ("zfp", torch.float32, 4096, 1024, 1024, 16, 2, 1.0)
    for train in (False, True):
        _compare(_run(True, *args, train), _run(False, *args, train), 1e-3)


# A token that is not finite is lost, the others are not: same outputs as beside a row of zeros, the same gradients of theirs.  Up to 32 tokens (the gate sends the
# rows itself) and more; as one node and by its steps
@pytest.mark.parametrize("codec,dtype", [("no", torch.bfloat16), ("int8", torch.bfloat16), ("no", torch.float32), ("int8", torch.float32), ("zfp", torch.float32),
                                         ("lz", torch.float32)])
@pytest.mark.parametrize("T,E,k", [(4, 8, 2), (32, 4, 3), (33, 8, 2), (300, 16, 2)])
@pytest.mark.parametrize("native", [True, False])
def test_layer_with_tokens_that_are_not_finite(native, T, E, k, codec, dtype):
    from planmoe_amd import overlap
    print("case", native, T, E, k, codec, dtype, flush=True)
    overlap.NATIVE_LAYER = native
    try:
        layer = _layer(dtype, codec, M=128, H=256, E=E)
        g = torch.Generator(device=DEV).manual_seed(T)
        x, gy = (torch.randn(T, 128, device=DEV, generator=g).to(dtype) for _ in range(2))
        lost = torch.arange(T, device=DEV) % 4 == 1
        outs = []
        for value in (0.0, float("nan"), float("inf")):
            v = x.clone()
            v[lost] = 0.0
            v[lost, 3] = value
            v.requires_grad_(True)
            y = layer(v, top_k=k)
            y.backward(gy)
            torch.cuda.synchronize()
            outs.append((y.detach(), v.grad))
            layer.zero_grad(set_to_none=True)
    finally:
        overlap.NATIVE_LAYER = True
    for y, dx in outs[1:]:
        assert bool(y[lost].isnan().any())
        if codec in ("no", "int8"):               # (a block of the other codecs holds rows of several tokens)
            assert torch.equal(y[~lost], outs[0][0][~lost]) and bool(y[~lost].isfinite().all()) and torch.equal(dx[~lost], outs[0][1][~lost])


# The second product left in shares of its reduction, which the combine adds.  Rows against 64 bits: the sum and the biased sum are each rounded to
# bf16 (2^-9 of them), the fp32 sums before it are off by at most H 2^-23 of the sum of magnitudes; everything behind the rows against the general
# path on those rows, bit for bit.  Few rows (up to 16, up to 32) and tiles; fewer pairs than experts, one share; a last share that is shorter;
# columns that are no whole tiles; one, two and three choices; capacities that drop; rows of 520 and 4096 values; an expert without a row.
@pytest.mark.parametrize("T,M,H,E,k,cap,skewed", [
    (1, 4096, 1024, 8, 2, 4, False), (2, 4096, 1024, 8, 2, 4, False), (1, 1032, 2056, 8, 1, 4, False), (8, 1024, 4096, 8, 2, 4, True), (7, 520, 1032, 4, 3, 16, False),
    (30, 264, 2048, 4, 2, 24, True), (60, 520, 1032, 4, 2, 40, False), (200, 1024, 4096, 8, 2, 64, True), (333, 136, 520, 3, 3, 129, True),
    (150, 4096, 576, 1, 1, 140, False), (90, 1000, 2000, 2, 1, 64, False)])
@pytest.mark.parametrize("with_bias", [True, False])
def test_product_in_shares_and_combine(T, M, H, E, k, cap, skewed, with_bias):
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    print("case", T, M, H, E, k, cap, skewed, with_bias, flush=True)
    g = torch.Generator(device=DEV).manual_seed(T + M + E)
    randn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    scores = randn(T, E)
    if skewed:
        scores[:, E - 1] += 3.0
        scores[:, 0] -= 9.0
    routed = ops.route_topk(torch.softmax(scores, 1), k)
    idx, loc, gates = routed["indices"].view(k, T), routed["locations"].view(k, T), routed["gates"].view(k, T).float()
    counts = torch.stack([torch.bincount(idx[j].long(), minlength=E) for j in range(k)]).int()
    h, w2 = randn(E, cap, H).bfloat16(), (randn(E, H, M) * H ** -0.5).bfloat16()
    b2 = randn(E, M).bfloat16() if with_bias else None
    hint = min(cap, (T * k + E - 1) // E)
    p, dt, st = ops._ptr, ops._dt(h, "t"), ops._stream(h)

    def run(codec, keep_rows, keep_codes):
        rows, out = torch.full((E, cap, M), 7.0, dtype=torch.bfloat16, device=DEV), torch.full((T, M), 7.0, dtype=torch.bfloat16, device=DEV)
        codes, mn, scale = (torch.zeros(E, cap, M, dtype=torch.uint8, device=DEV), torch.zeros(E, cap, dtype=torch.bfloat16, device=DEV),
                            torch.zeros(E, cap, dtype=torch.bfloat16, device=DEV)) if keep_codes else (None, None, None)
        size = lib.planmoe_layer_product_combine_workspace_bytes(dt, codec, H, k, T, M, E, cap, hint)
        assert size > 0 and size % (E * cap * M * 4) == 0
        ws = torch.full((size // 4,), float("nan"), device=DEV)
        check(lib.planmoe_layer_product_combine(p(h), p(w2), p(b2), dt, codec, H, p(gates), p(idx), p(loc), T, k, T, M, E, cap, p(counts), 1, hint, p(rows),
                                                int(keep_rows), p(codes), p(mn), p(scale), p(out), p(ws), size, st))
        return rows, out, codes, mn, scale

    rows, out = run(0, True, False)[:2]
    alone, again = run(0, False, False)[:2]
    torch.cuda.synchronize()
    bits = lambda t: t.view(torch.int16)
    assert torch.equal(bits(out), bits(again)) and bool((alone == 7.0).all())
    used = (torch.arange(cap, device=DEV)[None] < counts.sum(0)[:, None])
    assert bool((rows[~used] == 7.0).all())
    exact = h.double() @ w2.double()
    size = h.double().abs() @ w2.double().abs()
    want = exact + (b2.double()[:, None] if with_bias else 0.0)
    bound = exact.abs() * 2.0 ** -8 + want.abs() * 2.0 ** -8 + size * H * 2.0 ** -23 + 1e-30
    assert bool(((rows.double() - want).abs() <= bound)[used].all())
    check(lib.planmoe_layer_combine(p(rows), dt, 0, p(gates), p(idx), p(loc), T, k, T, M, E, cap, p(again), st))
    assert torch.equal(bits(out), bits(again))
    _, out8, codes, mn, scale = run(1, False, True)
    plain8 = run(1, False, False)[1]
    want_codes, want_mn, want_scale = torch.zeros_like(codes), torch.zeros_like(mn), torch.zeros_like(scale)
    check(lib.planmoe_layer_combine_keep(p(rows), dt, p(gates), p(idx), p(loc), T, k, T, M, E, cap, p(again), p(want_codes), p(want_mn), p(want_scale), st))
    torch.cuda.synchronize()
    assert torch.equal(bits(out8), bits(again)) and torch.equal(bits(plain8), bits(again))
    assert torch.equal(codes, want_codes) and torch.equal(mn, want_mn) and torch.equal(scale, want_scale)


# a capacity that leaves room for fewer shares than the eight that there would be
@pytest.mark.parametrize("T,M,H,E,k,cap,splits", [(64, 512, 2048, 4, 2, 2048, 4), (64, 512, 2048, 4, 2, 4096, 2)])
def test_product_in_fewer_shares(T, M, H, E, k, cap, splits):
    from planmoe_amd._lib import lib
    hint = min(cap, (T * k + E - 1) // E)
    assert lib.planmoe_layer_product_combine_workspace_bytes(1, 0, H, k, T, M, E, cap, hint) == splits * E * cap * M * 4
    assert lib.planmoe_layer_product_combine_workspace_bytes(1, 0, H, k, T, M, E, cap // 2, hint) == 2 * splits * E * (cap // 2) * M * 4
    test_product_in_shares_and_combine(T, M, H, E, k, cap, False, True)


# The combine that adds the gate's share of the gradient of x, for 9 to 16 experts: against the combine as it is and the product in 64 bits.  One token,
# an odd number (two a wave in fp32), rows of one piece, of one more than a wave's 64 and of 8 KB; choices without a slot
@pytest.mark.parametrize("T,M,E,k,cap", [(1, 8, 9, 1, 1), (5, 520, 16, 2, 1), (301, 1032, 11, 3, 40), (64, 2048, 16, 2, 8), (33, 4096, 16, 2, 4),
                                         (1281, 1032, 12, 2, 200), (2049, 264, 16, 1, 100)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("codec", [0, 1])
def test_layer_dx_of_up_to_16_experts(T, M, E, k, cap, dtype, codec):
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    if dtype == torch.float32 and M > 2048:
        pytest.skip("rows of up to 8 KB")
    print("case", T, M, E, k, cap, dtype, codec, flush=True)
    g = torch.Generator(device=DEV).manual_seed(T + M + E)
    routed = ops.route_topk(torch.softmax(torch.randn(T, E, generator=g, device=DEV), 1), k)
    idx, loc = routed["indices"].view(k, T), routed["locations"].view(k, T)
    rows, wg = torch.randn(E * cap, M, generator=g, device=DEV).to(dtype), torch.randn(E, M, generator=g, device=DEV).to(dtype)
    gl = torch.randn(T, E, generator=g, device=DEV)
    out, plain = torch.empty(T, M, dtype=dtype, device=DEV), torch.empty(T, M, dtype=dtype, device=DEV)
    p, dt, st = ops._ptr, ops._dt(rows, "t"), ops._stream(rows)
    check(lib.planmoe_layer_dx(p(rows), dt, codec, p(idx), p(loc), T, k, T, M, E, cap, p(gl), p(wg), p(out), st))
    check(lib.planmoe_layer_combine(p(rows), dt, codec, None, p(idx), p(loc), T, k, T, M, E, cap, p(plain), st))
    torch.cuda.synchronize()
    share, size = gl.to(dtype).double() @ wg.double(), gl.to(dtype).double().abs() @ wg.double().abs() + plain.double().abs()
    want = plain.double() + share
    # E + 1 terms in fp32, then one rounding
    bound = want.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) + size * (E + 1) * 2.0 ** -24 + 1e-30
    assert bool(((out.double() - want).abs() <= bound).all())


# Few tokens, up to 8 experts: the same bits as the combine and the gate's share in launches of their own.  One token, an odd number; rows of less than a
# wave's 64 pieces, of one more, of two, five and nine times 64 and of sixteen, the widest; the last number of tokens that is few and the first that is not
@pytest.mark.parametrize("T,M,E,k,cap", [(1, 8, 1, 1, 1), (5, 264, 8, 2, 1), (255, 520, 3, 2, 100), (37, 1288, 8, 2, 8), (131, 2568, 5, 3, 64), (9, 4096, 8, 2, 4), (7, 8192, 4, 2, 4),
                                         (256, 3080, 2, 1, 100), (257, 3080, 2, 1, 100), (768, 776, 8, 2, 200), (769, 776, 8, 2, 200), (4096, 264, 4, 1, 1000), (4097, 264, 4, 1, 1000),
                                         (512, 776, 8, 2, 100), (513, 776, 8, 2, 100), (1024, 264, 8, 2, 300), (1025, 264, 8, 2, 300), (1280, 1032, 8, 2, 300), (1281, 1032, 8, 2, 300),
                                         (1536, 2568, 4, 1, 500), (1537, 2568, 4, 1, 500), (3072, 4104, 2, 1, 2000), (3073, 4104, 2, 1, 2000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("codec", [0, 1])
def test_layer_dx_of_few_tokens(T, M, E, k, cap, dtype, codec):
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    if dtype == torch.float32 and M > 4096:
        pytest.skip("rows of up to 16 KB")
    print("case", T, M, E, k, cap, dtype, codec, flush=True)
    g = torch.Generator(device=DEV).manual_seed(T + M + E)
    routed = ops.route_topk(torch.softmax(torch.randn(T, E, generator=g, device=DEV), 1), k)
    idx, loc = routed["indices"].view(k, T), routed["locations"].view(k, T)
    rows, wg = torch.randn(E * cap, M, generator=g, device=DEV).to(dtype), torch.randn(E, M, generator=g, device=DEV).to(dtype)
    rows[0] = float("inf")                   # (what a choice without a slot reads and does not use)
    gl = torch.randn(T, E, generator=g, device=DEV)
    out, want = torch.empty(T, M, dtype=dtype, device=DEV), torch.empty(T, M, dtype=dtype, device=DEV)
    p, dt, st = ops._ptr, ops._dt(rows, "t"), ops._stream(rows)
    check(lib.planmoe_layer_dx(p(rows), dt, codec, p(idx), p(loc), T, k, T, M, E, cap, p(gl), p(wg), p(out), st))
    check(lib.planmoe_layer_combine(p(rows), dt, codec, None, p(idx), p(loc), T, k, T, M, E, cap, p(want), st))
    check(lib.planmoe_gate_dx_accumulate(p(want), dt, p(gl), p(wg), T, M, E, st))
    torch.cuda.synchronize()
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    same = (out.view(bits) == want.view(bits)) | (out.isnan() & want.isnan())
    assert bool(same.all())
