"""The routing API's nodes (csrc/ext/routing.cpp) against the step-by-step classes: the same kernels in the same order,
so everything is equal bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _fresh(*tensors):
    return [t.detach().clone().requires_grad_(t.is_floating_point()) for t in tensors]


# one choice, more choices than a plane's neighbours, one token; planes of one buffer and planes that lie apart
@pytest.mark.parametrize("T,M,E,k", [(1, 8, 4, 1), (77, 24, 5, 3), (300, 130, 3, 2)])
@pytest.mark.parametrize("postscore", [True, False])
@pytest.mark.parametrize("apart", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_nodes_equal_the_steps(T, M, E, k, postscore, apart, dtype):
    import planmoe_amd as pm
    from planmoe_amd import fast_dispatch as fd
    print("case", T, M, E, k, postscore, apart, dtype, flush=True)
    g = torch.Generator().manual_seed(T + M)
    scores = torch.softmax(torch.randn(T, E, generator=g), 1).to(DEV)
    x, gy = (torch.randn(T, M, generator=g).to(dtype).to(DEV) for _ in range(2))

    def steps(s, v):
        gates, loss, idx, loc, _ = fd.route(s, k)
        cap = fd.ops.capacity(T, E, k, 1.0, 4)
        d = fd.fast_dispatcher(E, cap, M, dtype)
        d.update(list(idx), list(loc), list(gates), cap, is_postscore=postscore)
        slots = fd.GatingEncoder.apply(d, v, *([] if postscore else d.gates_))
        return slots, fd.GatingDecoder.apply(d, slots, *(d.gates_ if postscore else [])), loss

    def nodes(s, v):
        crit, loss = pm.extract_critical(s, k, alignment=4)
        if apart:
            crit = (crit[0],) + tuple([t.clone() for t in part] for part in crit[1:4]) + crit[4:]
        slots = pm.fast_encode(v, crit, is_postscore=postscore)
        return slots, pm.fast_decode(slots, crit, is_postscore=postscore), loss

    got = []
    for f in (steps, nodes):
        s, v = _fresh(scores, x)
        slots, y, loss = f(s, v)
        torch.autograd.backward([y, loss], [gy, torch.full_like(loss, 0.5)])
        torch.cuda.synchronize()
        got.append((slots.detach().reshape(-1, M), y.detach(), loss.detach(), v.grad, s.grad))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_gradients_that_are_not_asked_for():
    import planmoe_amd as pm
    T, M, E = 64, 16, 4
    scores, x = torch.rand(T, E, device=DEV), torch.randn(T, M, device=DEV)
    crit, loss = pm.extract_critical(scores, 2)
    assert not loss.requires_grad and not crit[3][0].requires_grad
    v = x.clone().requires_grad_()
    pm.fast_decode(pm.fast_encode(v, crit), crit).sum().backward()
    assert v.grad is not None
    s = scores.clone().requires_grad_()
    crit, loss = pm.extract_critical(s, 2, loss_fn=None)
    assert loss is None
    crit[3][1].sum().backward()                  # one choice's gates only
    want = s.grad
    s2 = scores.clone().requires_grad_()
    gates = pm.fast_dispatch.route(s2, 2)[0]
    gates[1].sum().backward()
    torch.cuda.synchronize()
    assert torch.equal(want, s2.grad)


def test_the_backward_pass_reads_the_planes_where_they_are_then():
    """A choice's indices exchanged for a copy elsewhere (as an optimizer or a memory saver does with .data) between the
    forward and the backward pass: the planes are not where the forward pass found them, nor equally far apart."""
    import planmoe_amd
    g = torch.Generator().manual_seed(5)
    scores = torch.softmax(torch.randn(70, 6, generator=g), 1).to(DEV)
    x, grad = torch.randn(70, 40, generator=g).to(DEV), torch.randn(70, 40, generator=g).to(DEV)

    def run(exchange):
        xs = x.clone().requires_grad_(True)
        crit, _ = planmoe_amd.extract_critical(scores, 2, capacity_factor=1.0, alignment=4)
        y = planmoe_amd.fast_decode(planmoe_amd.fast_encode(xs, crit), crit)
        if exchange:
            crit[1][0].data = crit[1][0].data.clone()
        y.backward(grad)
        torch.cuda.synchronize()
        return y.detach(), xs.grad

    (y0, g0), (y1, g1) = run(False), run(True)
    assert torch.equal(y0, y1) and torch.equal(g0, g1)


@pytest.mark.parametrize("k", [1, 2])
def test_index_planes_edited_in_place_are_refused(k):
    """The gradient reads the indices again, so a plane edited between the forward and the backward pass would change it
    without a word: autograd refuses it (the edits here stay in range).  The slots are not read: they may be edited."""
    import planmoe_amd
    g = torch.Generator().manual_seed(11)
    scores = torch.softmax(torch.randn(50, 6, generator=g), 1).to(DEV)

    def run(plane):
        s = scores.clone().requires_grad_(True)
        crit, loss = planmoe_amd.extract_critical(s, k, alignment=4)
        if plane is not None:
            crit[plane][-1].zero_()
        (crit[3][0].sum() + loss).backward()
        torch.cuda.synchronize()
        return s.grad

    want = run(None)
    assert torch.equal(run(2), want)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        run(1)


@pytest.mark.parametrize("postscore", [True, False])
def test_nodes_on_a_stream_of_their_own(postscore):
    """The forward pass on another stream, behind work that is still running there; the backward pass asked for from the
    stream that was current before."""
    import planmoe_amd as pm
    g = torch.Generator().manual_seed(9)
    scores = torch.softmax(torch.randn(300, 6, generator=g), 1).to(DEV)
    x, gy = torch.randn(300, 40, generator=g).to(DEV), torch.randn(300, 40, generator=g).to(DEV)

    def run(s, v):
        crit, loss = pm.extract_critical(s, 2, alignment=4)
        return pm.fast_decode(pm.fast_encode(v, crit, is_postscore=postscore), crit, is_postscore=postscore), loss

    s, v = _fresh(scores, x)
    y, loss = run(s, v)
    torch.autograd.backward([y, loss], [gy, torch.full_like(loss, 0.5)])
    want = [y.detach(), loss.detach(), s.grad, v.grad]
    s, v, stream = torch.zeros_like(scores).requires_grad_(True), torch.zeros_like(x).requires_grad_(True), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        torch.cuda._sleep(20_000_000)            # (about 10 ms: what does not wait for the copies below sees other values)
        with torch.no_grad():
            s.copy_(scores)
            v.copy_(x)
        y, loss = run(s, v)
    torch.autograd.backward([y, loss], [gy, torch.full_like(loss, 0.5)])
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    for a, b in zip(want, [y.detach(), loss.detach(), s.grad, v.grad]):
        assert torch.equal(a, b)
