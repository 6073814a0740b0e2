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
    assert seen and overlap.native_codec(layer, layer.gates[0], x, 1, 1, 4) is None
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
