"""planmoe_expert_gemm / planmoe_expert_gemm_relu_bwd (the experts' products, bf16 and fp32, with row counts)
and the two column reductions of the layer's backward pass, against fp64 on the host.

Tolerances: fp32 sums of n terms are within (n + 2) 2^-24 of the sum of their magnitudes, whatever their
order; a bf16 result adds 2^-8 of itself (half an ulp is 2^-9)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _bound(ref, mag, terms, dtype):
    return (terms + 2) * 2.0 ** -24 * mag + (2.0 ** -8 * ref.abs() if dtype == torch.bfloat16 else 0.0) + 1e-30


# sizes one piece either side of 256 and 128 and of k-tiles of 64 (bf16) and 32 (fp32), one k-tile, an odd number of them, more than eight tile columns, one row
# (products as small as these go to the kernels for few rows and few tiles: test_expert_gemm_in_every_kernel has the others)
SHAPES = [(1, 1, 8, 8), (2, 127, 136, 64), (3, 129, 264, 72), (2, 255, 520, 136), (2, 257, 128, 200), (1, 300, 2312, 64), (5, 40, 256, 320)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["nn", "nt", "tn"])
@pytest.mark.parametrize("B,m,n,k", SHAPES)
def test_expert_gemm_against_fp64(B, m, n, k, form, dtype):
    from planmoe_amd import ops
    if form == "tn":
        m = (m + 7) // 8 * 8                     # the fast index of a
    print("case", form, dtype, B, m, n, k, flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(*((B, k, m) if form == "tn" else (B, m, k)), generator=g).to(dtype)
    b = torch.randn(*((B, n, k) if form == "nt" else (B, k, n)), generator=g).to(dtype)
    with_bias = form == "nn"
    bias = torch.randn(B, n, generator=g).to(dtype) if with_bias else None
    got = ops.expert_gemm(form, a.to(DEV), b.to(DEV), bias.to(DEV) if with_bias else None, relu=with_bias)
    torch.cuda.synchronize()
    ad, bd = a.double(), b.double()
    ad, bd = (ad.transpose(1, 2) if form == "tn" else ad), (bd.transpose(1, 2) if form == "nt" else bd)
    ref, mag = ad @ bd, ad.abs() @ bd.abs()
    tol = _bound(ref, mag, k, dtype)
    if with_bias:
        ref, tol = ref + bias.double()[:, None, :], tol + _bound(ref + bias.double()[:, None, :], bias.double().abs()[:, None, :], 1, dtype)
        ref = ref.clamp(min=0)                   # (clamping both sides of a comparison cannot move them apart)
    assert bool(((got.double().cpu() - ref).abs() <= tol).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,cap,n,k,hint", [(4, 200, 264, 136, 0), (6, 520, 520, 64, 100), (64, 20, 72, 72, 5)])
def test_expert_gemm_takes_the_rows_in_use_only(B, cap, n, k, hint, dtype):
    """Row counts from two planes, rounded up to 1 and 4: none, few, more than the capacity; rows of the operands beyond
    them hold NaN, rows of the result beyond them keep what was there; a tn product sums over the rows in use."""
    from planmoe_amd import ops
    g = torch.Generator().manual_seed(B + cap)
    live = torch.randint(0, cap, (2, B), generator=g, dtype=torch.int32) // 2
    live[:, 0] = 0
    live[:, 1] = cap
    live[0, 2], live[1, 2] = 1, 0
    for rnd in (1, 4):
        rows = [min(cap, (int(c) + rnd - 1) // rnd * rnd) for c in live.sum(0)]
        a = torch.randn(B, cap, k, generator=g).to(dtype)
        w = torch.randn(B, k, n, generator=g).to(dtype)
        dy = torch.randn(B, cap, n, generator=g).to(dtype)
        for e, r in enumerate(rows):
            a[e, r:] = float("nan")
            dy[e, r:] = float("nan")
        out = torch.full((B, cap, n), 7.0, dtype=dtype, device=DEV)
        ops.expert_gemm("nn", a.to(DEV), w.to(DEV), None, live=live.to(DEV), live_round=rnd, rows_hint=hint, out=out)
        dw = ops.expert_gemm("tn", a.to(DEV), dy.to(DEV), live=live.to(DEV), live_round=rnd, rows_hint=hint)
        torch.cuda.synchronize()
        out, dw = out.cpu(), dw.cpu()
        for e, r in enumerate(rows):
            x, d = a[e, :r].double(), dy[e, :r].double()
            ref, mag = x @ w[e].double(), x.abs() @ w[e].double().abs()
            assert bool(((out[e, :r].double() - ref).abs() <= _bound(ref, mag, k, dtype)).all()), (e, r)
            assert bool((out[e, r:] == 7.0).all()), (e, r)
            ref, mag = x.t() @ d, x.abs().t() @ d.abs()
            assert bool(((dw[e].double() - ref).abs() <= _bound(ref, mag, cap, dtype)).all()), (e, r)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,m,n,k,counted", [(2, 130, 136, 72, False), (3, 300, 520, 128, True), (1, 8, 8, 8, False)])
def test_expert_gemm_relu_backward_and_its_bias_gradient(B, m, n, k, counted, dtype):
    from planmoe_amd import ops
    g = torch.Generator().manual_seed(m + n)
    dy, w = torch.randn(B, m, k, generator=g).to(dtype), torch.randn(B, n, k, generator=g).to(dtype)
    h = torch.randn(B, m, n, generator=g).clamp(min=0).to(dtype)
    live = torch.tensor([[m // 2 + 3 * e for e in range(B)]], dtype=torch.int32) if counted else None
    got, db = ops.expert_gemm_relu_bwd(dy.to(DEV), w.to(DEV), h.to(DEV), live=live.to(DEV) if counted else None)
    torch.cuda.synchronize()
    got, db = got.cpu(), db.cpu()
    for e in range(B):
        r = min(m, int(live[0, e])) if counted else m
        ref, mag = dy[e, :r].double() @ w[e].double().t(), dy[e, :r].double().abs() @ w[e].double().abs().t()
        keep = h[e, :r] > 0
        assert bool(((got[e, :r].double() - ref * keep).abs() <= _bound(ref, mag, k, dtype)).all())
        stored = got[e, :r].double()             # the sums are of what was stored
        tol = _bound(stored.sum(0), stored.abs().sum(0), r, dtype)
        assert bool(((db[e].double() - stored.sum(0)).abs() <= tol).all())


# few rows per expert against a whole weight: one row, either side of 16, 32 and 64 rows; columns and reduction lengths that
# are and are not whole steps of the waves that share a reduction
@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(8, 8), (136, 520), (264, 1032), (64, 4096)])
def test_expert_gemm_with_few_rows(m, n, k):
    from planmoe_amd import ops
    print("case", m, n, k, flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    B, dtype = 3, torch.bfloat16
    live = torch.tensor([[m, 0, max(m // 2, 1)]], dtype=torch.int32)
    a, bias = torch.randn(B, m, k, generator=g).to(dtype), torch.randn(B, n, generator=g).to(dtype)
    w, h = torch.randn(B, k, n, generator=g).to(dtype), torch.randn(B, m, n, generator=g).clamp(min=0).to(dtype)
    for e in range(B):
        a[e, int(live[0, e]):] = float("nan")
    wt = w.transpose(1, 2).contiguous()
    nn = torch.full((B, m, n), 7.0, dtype=dtype, device=DEV)
    nt, masked = nn.clone(), nn.clone()
    ops.expert_gemm("nn", a.to(DEV), w.to(DEV), bias.to(DEV), relu=True, live=live.to(DEV), out=nn)
    ops.expert_gemm("nt", a.to(DEV), wt.to(DEV), live=live.to(DEV), out=nt)
    _, db = ops.expert_gemm_relu_bwd(a.to(DEV), wt.to(DEV), h.to(DEV), live=live.to(DEV), out=masked)
    torch.cuda.synchronize()
    nn, nt, masked, db = nn.cpu().double(), nt.cpu().double(), masked.cpu().double(), db.cpu().double()
    for e in range(B):
        r = int(live[0, e])
        ref, mag = a[e, :r].double() @ w[e].double(), a[e, :r].double().abs() @ w[e].double().abs()
        tol = _bound(ref, mag, k, dtype)
        biased = ref + bias[e].double()
        assert bool(((nn[e, :r] - biased.clamp(min=0)).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, dtype)).all())
        assert bool(((nt[e, :r] - ref).abs() <= tol).all())
        assert bool(((masked[e, :r] - ref * (h[e, :r] > 0)).abs() <= tol).all())
        assert bool((nn[e, r:] == 7.0).all()) and bool((nt[e, r:] == 7.0).all()) and bool((masked[e, r:] == 7.0).all())
        stored = masked[e, :r]
        assert bool(((db[e] - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), max(r, 1), dtype)).all())


# weights of 16 MB and more, read past the caches: 32 columns a work-group (99 and 195 of them: the last are no whole sixteen), 64 and 128;
# rows either side of a fragment, a reduction whose last step is partial
@pytest.mark.parametrize("m", [1, 16, 17, 32])
@pytest.mark.parametrize("B,n,k", [(3, 1032, 4104), (3, 2072, 2056), (3, 4104, 1032), (5, 8200, 520)])
def test_expert_gemm_with_few_rows_of_large_weights(m, B, n, k):
    from planmoe_amd import ops
    print("case", m, B, n, k, flush=True)
    assert B * n * k * 2 >= 16 << 20
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    dtype = torch.bfloat16
    randn = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    rows = [m, 0, max(m // 2, 1), m, 1][:B]
    a, bias, w, h = randn(B, m, k), randn(B, n), randn(B, k, n), randn(B, m, n).clamp(min=0)
    for e in range(B):
        a[e, rows[e]:] = float("nan")
    live = torch.tensor([rows], dtype=torch.int32, device=DEV)
    wt = w.transpose(1, 2).contiguous()
    nn = torch.full((B, m, n), 7.0, dtype=dtype, device=DEV)
    nt, masked = nn.clone(), nn.clone()
    ops.expert_gemm("nn", a, w, bias, relu=True, live=live, out=nn)
    ops.expert_gemm("nt", a, wt, live=live, out=nt)
    _, db = ops.expert_gemm_relu_bwd(a, wt, h, live=live, out=masked)
    torch.cuda.synchronize()
    for e, r in enumerate(rows):
        x, y = a[e, :r].double(), w[e].double()
        ref, mag = x @ y, x.abs() @ y.abs()
        tol, biased = _bound(ref, mag, k, dtype), ref + bias[e].double()
        assert bool(((nn[e, :r].double() - biased.clamp(min=0)).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, dtype)).all())
        assert bool(((nt[e, :r].double() - ref).abs() <= tol).all())
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all())
        assert bool((nn[e, r:] == 7.0).all()) and bool((nt[e, r:] == 7.0).all()) and bool((masked[e, r:] == 7.0).all())
        stored = masked[e, :r].double()
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), max(r, 1), dtype)).all())


# 256 work-groups that stay take 256 x 256 tiles, four to a tile row here; what is left for a last round is a launch of
# quarters up to 128 tiles.  Rows in use that leave 0, 4 (one row of the last tile), 128 and 132 tiles, and fewer than one round
# (with k = 4096 and 8192 rows a batch expected; with k = 512 what is picked for the rows that are there)
@pytest.mark.parametrize("rows", [16384, 16385, 24576, 24577, 300])
@pytest.mark.parametrize("k", [512, 4096])
def test_expert_gemm_last_round(rows, k):
    from planmoe_amd import ops
    print("case", rows, k, flush=True)
    cap, n, dtype = 24832, 1024, torch.bfloat16
    hint = 8192 if k == 4096 else rows // 2
    kernels = [ops.expert_gemm_kernel(form, dtype, 2, cap // 2, n, k, counted=True, rows_hint=hint) for form in ("nn", "nt")]
    assert kernels == ["256x256 and quarters" if k == 4096 else {150: "128x128 alone", 8192: "160x256", 12288: "256x256"}[rows // 2]] * 2
    g = torch.Generator(device=DEV).manual_seed(rows)
    a, w = torch.randn(2, cap // 2, k, device=DEV, generator=g).to(dtype), torch.randn(2, k, n, device=DEV, generator=g).to(dtype)
    first = 0 if rows < 512 else rows // 512 * 256          # (the odd row is the second batch's)
    live = torch.tensor([[first, rows - first]], dtype=torch.int32, device=DEV)
    h = torch.randn(2, cap // 2, n, device=DEV, generator=g).clamp(min=0).to(dtype)
    out = torch.full((2, cap // 2, n), 7.0, dtype=dtype, device=DEV)
    masked = out.clone()
    ops.expert_gemm("nn", a, w, live=live, out=out, rows_hint=hint)
    _, db = ops.expert_gemm_relu_bwd(a, w.transpose(1, 2).contiguous(), h, live=live, out=masked, rows_hint=hint)
    torch.cuda.synchronize()
    for e in range(2):
        r = int(live[0, e])
        ref, mag = a[e, :r].double() @ w[e].double(), a[e, :r].double().abs() @ w[e].double().abs()
        tol = _bound(ref, mag, k, dtype)
        assert bool(((out[e, :r].double() - ref).abs() <= tol).all()), e
        assert bool((out[e, r:] == 7.0).all()), e
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all()), e
        assert bool((masked[e, r:] == 7.0).all()), e
        stored = masked[e, :r].double()
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), r, dtype)).all()), e


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,M,E", [(1, 8, 1), (33, 520, 3), (1000, 264, 9), (517, 2056, 16)])
def test_gate_weight_gradient_and_row_sums(T, M, E, dtype):
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    g = torch.Generator().manual_seed(T + M)
    x, gl = torch.randn(T, M, generator=g).to(dtype), torch.randn(T, E, generator=g)
    xd, gd = x.to(DEV), gl.to(DEV)
    dw = torch.empty(E, M, dtype=dtype, device=DEV)
    ws = torch.empty(lib.planmoe_gate_dw_workspace_bytes(T, M, E), dtype=torch.uint8, device=DEV)
    check(lib.planmoe_gate_dw(ops._ptr(xd), ops._dt(xd, "t"), ops._ptr(gd), T, M, E, ops._ptr(dw), ops._ptr(ws), ws.numel(), ops._stream(xd)))
    live = torch.tensor([[T // 2], [T - T // 2 - T // 3]], dtype=torch.int32, device=DEV)
    out = torch.empty(1, M, dtype=dtype, device=DEV)
    ws2 = torch.empty(lib.planmoe_rows_colsum_workspace_bytes(1, T, M), dtype=torch.uint8, device=DEV)
    check(lib.planmoe_rows_colsum(ops._ptr(xd), ops._dt(xd, "t"), 1, T, M, ops._ptr(live), 2, 4, ops._ptr(out), ops._ptr(ws2), ws2.numel(), ops._stream(xd)))
    torch.cuda.synchronize()
    gr = gl.to(dtype).double()
    ref, mag = gr.t() @ x.double(), gr.abs().t() @ x.double().abs()
    half = 2.0 ** -8 if dtype != torch.float32 else 0.0
    assert bool(((dw.double().cpu() - ref).abs() <= (T + 2) * 2.0 ** -24 * mag + half * ref.abs() + 1e-30).all())
    rows = x[:min(T, (T - T // 3 + 3) // 4 * 4)].double()
    assert bool(((out[0].double().cpu() - rows.sum(0)).abs() <= (T + 2) * 2.0 ** -24 * rows.abs().sum(0) + half * rows.sum(0).abs() + 1e-30).all())


# Rows that end on a tile of 256 or 128 and just behind one, batches of less than a tile and of no rows, in tiles of 160 rows and in those of 256 with
# their last round in quarters: a quarter that has no rows stores nothing; several tiles for a work-group; some have no row counts
@pytest.mark.parametrize("kernel,n,k,hint,counts", [
    ("160x256", 1024, 512, 4096, [4096, 4097, 4160, 4161]), ("160x256", 1024, 512, 4096, [4224, 4225, 128, 1]),
    ("160x256", 2048, 2048, 500, [512, 513, 576, 577, 500, 64, 1, 0]), ("160x256", 1024, 1024, 0, [4160] * 4),
    ("256x256 and quarters", 1024, 4096, 4096, [4096, 4097, 4160, 4161, 4095, 4224, 4225, 4100]),
    ("256x256 and quarters", 1024, 4096, 4096, [4352, 4353, 4225, 1, 4224, 128, 4097, 0]), ("256x256 and quarters", 1016, 4104, 0, [4160] * 8)])
def test_expert_gemm_rows_around_a_tile(kernel, n, k, hint, counts):
    from planmoe_amd import ops
    print("case", kernel, n, k, counts, flush=True)
    B, cap, dtype = len(counts), max(counts) + (64 if hint else 0), torch.bfloat16
    assert all(ops.expert_gemm_kernel(form, dtype, B, cap, n, k, counted=bool(hint), rows_hint=hint) == kernel for form in ("nn", "nt"))
    g = torch.Generator(device=DEV).manual_seed(sum(counts))
    a, w = torch.randn(B, cap, k, device=DEV, generator=g).to(dtype), torch.randn(B, k, n, device=DEV, generator=g).to(dtype)
    bias, h = torch.randn(B, n, device=DEV, generator=g).to(dtype), torch.randn(B, cap, n, device=DEV, generator=g).clamp(min=0).to(dtype)
    live = torch.tensor([counts], dtype=torch.int32, device=DEV) if hint else None
    out = torch.full((B, cap, n), 7.0, dtype=dtype, device=DEV)
    masked = out.clone()
    ops.expert_gemm("nn", a, w, bias, relu=True, live=live, out=out, rows_hint=hint)
    _, db = ops.expert_gemm_relu_bwd(a, w.transpose(1, 2).contiguous(), h, live=live, out=masked, rows_hint=hint)
    torch.cuda.synchronize()
    for e, r in enumerate(counts):
        ref, mag = a[e, :r].double() @ w[e].double(), a[e, :r].double().abs() @ w[e].double().abs()
        tol, biased = _bound(ref, mag, k, dtype), ref + bias[e].double()
        assert bool(((out[e, :r].double() - biased.clamp(min=0)).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, dtype)).all()), e
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all()), e
        assert bool((out[e, r:] == 7.0).all()) and bool((masked[e, r:] == 7.0).all()), e
        stored = masked[e, :r].double()
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), max(r, 1), dtype)).all()), e


# fp32: few rows are served by waves on their own, whose sums take the reduction in the tiles' order: the first
# rows of a product do not depend on how many rows there are.  Either side of 16 and 32 rows, k steps and columns that are not whole
@pytest.mark.parametrize("m", [1, 16, 17, 32, 33])
@pytest.mark.parametrize("n,k", [(4, 4), (68, 20), (136, 520), (1104, 132)])
def test_expert_gemm_fp32_does_not_depend_on_the_number_of_rows(m, n, k):
    from planmoe_amd import ops
    print("case", m, n, k, flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    B, many = 2, 16384                           # (the many rows: 128 x 128 tiles)
    live = torch.tensor([[m, m // 2]], dtype=torch.int32)
    a, w, bias = torch.randn(B, many, k, generator=g).to(DEV), torch.randn(B, k, n, generator=g), torch.randn(B, n, generator=g).to(DEV)
    wt, w, few = w.transpose(1, 2).contiguous().to(DEV), w.to(DEV), a[:, :m].clone()
    h = torch.randn(B, m, n, generator=g).clamp(min=0)
    for e in range(B):
        few[e, int(live[0, e]):] = float("nan")
    nn, nt = torch.full((B, m, n), 7.0, device=DEV), torch.full((B, m, n), 7.0, device=DEV)
    masked = nn.clone()
    ops.expert_gemm("nn", few, w, bias, relu=True, live=live.to(DEV), out=nn)
    ops.expert_gemm("nt", few, wt, live=live.to(DEV), out=nt)
    _, db = ops.expert_gemm_relu_bwd(few, wt, h.to(DEV), live=live.to(DEV), out=masked)
    want_nn, want_nt = ops.expert_gemm("nn", a, w, bias, relu=True), ops.expert_gemm("nt", a, wt)
    torch.cuda.synchronize()
    for e in range(B):
        r = int(live[0, e])
        assert torch.equal(nn[e, :r], want_nn[e, :r]) and torch.equal(nt[e, :r], want_nt[e, :r])
        assert torch.equal(masked[e, :r], torch.where(h[e, :r].to(DEV) > 0, want_nt[e, :r], torch.zeros((), device=DEV)))
        assert bool((nn[e, r:] == 7.0).all()) and bool((nt[e, r:] == 7.0).all()) and bool((masked[e, r:] == 7.0).all())
        stored = masked[e, :r].double()
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), max(r, 1), torch.float32)).all())


# more rows than 256 (or 128) of them would fit in 2 GiB if they were as long: rows are no row length.  nn and nt rows,
# a tn product's reduction, the masked product
@pytest.mark.parametrize("dtype,rows", [(torch.float32, 2097160), (torch.float32, 4194312), (torch.bfloat16, 4194312)])
def test_expert_gemm_takes_millions_of_rows(dtype, rows):
    from planmoe_amd import ops
    print("case", dtype, rows, flush=True)
    n = k = 8
    g = torch.Generator(device=DEV).manual_seed(rows)
    a, dy = torch.randn(1, rows, k, device=DEV, generator=g).to(dtype), torch.randn(1, rows, n, device=DEV, generator=g).to(dtype)
    w, h = torch.randn(1, k, n, device=DEV, generator=g).to(dtype), torch.randn(1, rows, n, device=DEV, generator=g).clamp(min=0).to(dtype)
    ref, mag = a[0].double() @ w[0].double(), a[0].double().abs() @ w[0].double().abs()
    tol, wt = _bound(ref, mag, k, dtype), w.transpose(1, 2).contiguous()
    assert bool(((ops.expert_gemm("nn", a, w)[0].double() - ref).abs() <= tol).all())
    assert bool(((ops.expert_gemm("nt", a, wt)[0].double() - ref).abs() <= tol).all())
    masked, db = ops.expert_gemm_relu_bwd(a, wt, h)
    assert bool(((masked[0].double() - ref * (h[0] > 0)).abs() <= tol).all())
    stored = masked[0].double()
    assert bool(((db[0].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), rows, dtype)).all())
    got = ops.expert_gemm("tn", a, dy)[0].double()
    ref, mag = a[0].double().t() @ dy[0].double(), a[0].double().abs().t() @ dy[0].double().abs()
    assert bool(((got - ref).abs() <= _bound(ref, mag, rows, dtype)).all())
    # a few rows in use of many
    live = torch.tensor([[3]], dtype=torch.int32, device=DEV)
    out = torch.full((1, rows, n), 7.0, dtype=dtype, device=DEV)
    ops.expert_gemm("nn", a, w, live=live, rows_hint=3, out=out)
    ref = a[0, :3].double() @ w[0].double()
    torch.cuda.synchronize()
    assert bool(((out[0, :3].double() - ref).abs() <= tol[:3]).all()) and bool((out[0, 3:] == 7.0).all())


# few rows expected, many of an expert: the waves on their own find the row blocks in use among all batches.  Batches without
# rows first, last and in between, with one row, with a whole capacity; 64 batches; and no row counts at all
@pytest.mark.parametrize("B,cap,n,k,counted", [(5, 300, 68, 20, True), (64, 100, 132, 64, True), (3, 100, 260, 36, False), (1, 65, 64, 16, True)])
def test_expert_gemm_fp32_few_rows_expected_and_many_there(B, cap, n, k, counted):
    from planmoe_amd import ops
    print("case", B, cap, n, k, counted, flush=True)
    g = torch.Generator().manual_seed(B + cap)
    live = torch.randint(0, cap // 2, (2, B), generator=g, dtype=torch.int32)
    if B > 3:
        live[:, 0] = live[:, -1] = live[:, 2] = 0
        live[:, 1] = cap
        live[:, 3] = torch.tensor([0, 1])
    rows = [min(cap, int(c)) for c in live.sum(0)] if counted else [cap] * B
    a, h = torch.randn(B, cap, k, generator=g), torch.randn(B, cap, n, generator=g).clamp(min=0)
    w, bias = torch.randn(B, k, n, generator=g), torch.randn(B, n, generator=g)
    for e, r in enumerate(rows):
        a[e, r:] = float("nan")
    ad, wd, wt = a.to(DEV), w.to(DEV), w.transpose(1, 2).contiguous().to(DEV)
    kw = dict(live=live.to(DEV) if counted else None, rows_hint=3)
    nn = torch.full((B, cap, n), 7.0, device=DEV)
    nt, masked = nn.clone(), nn.clone()
    ops.expert_gemm("nn", ad, wd, bias.to(DEV), relu=True, out=nn, **kw)
    ops.expert_gemm("nt", ad, wt, out=nt, **kw)
    _, db = ops.expert_gemm_relu_bwd(ad, wt, h.to(DEV), out=masked, **kw)
    torch.cuda.synchronize()
    nn, nt, masked, db = nn.cpu().double(), nt.cpu().double(), masked.cpu().double(), db.cpu().double()
    for e, r in enumerate(rows):
        ref, mag = a[e, :r].double() @ w[e].double(), a[e, :r].double().abs() @ w[e].double().abs()
        tol, biased = _bound(ref, mag, k, torch.float32), ref + bias[e].double()
        assert bool(((nn[e, :r] - biased.clamp(min=0)).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, torch.float32)).all()), e
        assert bool(((nt[e, :r] - ref).abs() <= tol).all()), e
        assert bool(((masked[e, :r] - ref * (h[e, :r] > 0)).abs() <= tol).all()), e
        assert bool((nn[e, r:] == 7.0).all()) and bool((nt[e, r:] == 7.0).all()) and bool((masked[e, r:] == 7.0).all()), e
        stored = masked[e, :r]
        assert bool(((db[e] - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), max(r, 1), torch.float32)).all()), e


def _fp64(form, a, b):
    a, b = a.double(), b.double()
    a, b = (a.transpose(1, 2).contiguous() if form == "tn" else a), (b.transpose(1, 2).contiguous() if form == "nt" else b)
    return a @ b, a.abs() @ b.abs()


# fp32 on the bf16 matrix cores in three parts a value (six of the shapes; four run in 64 x 64 tiles with four k-tiles in LDS, and the same holds of them; every tile and form
# in parts is in test_expert_gemm_in_every_kernel): rows, columns and reductions that are no multiple of anything but 4, one past a tile and one
# k-tile's edge.  A k-slow operand's rows need not be a multiple of 4.
@pytest.mark.parametrize("form,B,m,n,k", [("nn", 8, 301, 712, 712), ("nt", 8, 299, 708, 700), ("tn", 8, 712, 716, 301), ("nn", 4, 999, 1004, 300),
                                          ("nt", 4, 1000, 1004, 292), ("tn", 4, 516, 2048, 1001), ("nn", 4, 2041, 1004, 260), ("nt", 16, 257, 1036, 1028),
                                          ("tn", 8, 1028, 1004, 129), ("tn", 8, 1028, 1024, 1)])
def test_expert_gemm_fp32_in_parts(form, B, m, n, k):
    from planmoe_amd import ops
    print("case", form, B, m, n, k, flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = torch.randn(*((B, k, m) if form == "tn" else (B, m, k)), device=DEV, generator=g)
    b = torch.randn(*((B, n, k) if form == "nt" else (B, k, n)), device=DEV, generator=g)
    got, (ref, mag) = ops.expert_gemm(form, a, b), _fp64(form, a, b)
    # six products of parts leave 2^-26 of a product out and are six sums for 16 k: inside the bound of k fp32 products and sums
    assert bool(((got.double() - ref).abs() <= _bound(ref, mag, k, torch.float32)).all())
    # parts of the smallest values are no subnormal bf16 values; sums that the scaled parts overflow are made again
    for scale_a, scale_b in ((2.0 ** -126, 1.0), (2.0 ** -63, 2.0 ** -62), (2.0 ** 100, 2.0 ** -100), (2.0 ** 60, 2.0 ** 55), (2.0 ** 125, 2.0 ** -120)):
        got, (ref, mag) = ops.expert_gemm(form, a * scale_a, b * scale_b), _fp64(form, a * scale_a, b * scale_b)
        # (a result below the normal range is rounded to 2^-149 in every sum)
        assert bool(((got.double() - ref).abs() <= _bound(ref, mag, k, torch.float32) - 1e-30 + (k + 2) * 2.0 ** -149).all()), (scale_a, scale_b)
    # infinities and NaN reach the results they belong to and no others
    a[0, 0, 7], a[B - 1, 0, 1] = float("inf"), float("nan")
    if k > 3:
        b[0, 2, 3], b[B - 1, 3, 2] = float("-inf"), 3.4e38
    got, (ref, mag) = ops.expert_gemm(form, a, b), _fp64(form, a, b)
    torch.cuda.synchronize()
    finite = ref.abs() < 3.4028235e38
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[got.isinf()], ref[got.isinf()].float()) and bool(got[finite].isfinite().all())
    assert bool(((got.double() - ref).abs()[finite] <= _bound(ref, mag, k, torch.float32)[finite]).all())


# the same with row counts: batches without rows and with a capacity's, rows beyond those in use hold NaN; the masked product and its sums
@pytest.mark.parametrize("B,cap,n,k,hint", [(16, 520, 1036, 1028, 500), (8, 320, 712, 716, 290), (4, 1100, 1004, 300, 980)])
def test_expert_gemm_fp32_in_parts_takes_the_rows_in_use_only(B, cap, n, k, hint):
    from planmoe_amd import ops
    print("case", B, cap, n, k, hint, flush=True)
    g = torch.Generator(device=DEV).manual_seed(B + cap)
    counts = [0, cap, 1, hint] + [cap // 2 + 7 * e for e in range(4, B)]
    live = torch.tensor([counts], dtype=torch.int32, device=DEV)
    a, dy = torch.randn(B, cap, k, device=DEV, generator=g), torch.randn(B, cap, n, device=DEV, generator=g)
    w, bias, h = torch.randn(B, k, n, device=DEV, generator=g), torch.randn(B, n, device=DEV, generator=g), torch.randn(B, cap, n, device=DEV, generator=g).clamp(min=0)
    rows = [min(cap, c) for c in counts]
    for e, r in enumerate(rows):
        a[e, r:] = dy[e, r:] = float("nan")
    nn = torch.full((B, cap, n), 7.0, device=DEV)
    masked = nn.clone()
    kw = dict(live=live, rows_hint=hint)
    ops.expert_gemm("nn", a, w, bias, out=nn, **kw)
    _, db = ops.expert_gemm_relu_bwd(a, w.transpose(1, 2).contiguous(), h, out=masked, **kw)
    dw = ops.expert_gemm("tn", a, dy, **kw)
    torch.cuda.synchronize()
    for e, r in enumerate(rows):
        x, wd = a[e, :r].double(), w[e].double()
        ref, mag = x @ wd, x.abs() @ wd.abs()
        tol, biased = _bound(ref, mag, k, torch.float32), ref + bias[e].double()
        assert bool(((nn[e, :r].double() - biased).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, torch.float32)).all()), e
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all()), e
        assert bool((nn[e, r:] == 7.0).all()) and bool((masked[e, r:] == 7.0).all()), e
        stored = masked[e, :r].double()
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), max(r, 1), torch.float32)).all()), e
        d = dy[e, :r].double()
        assert bool(((dw[e].double() - x.t() @ d).abs() <= _bound(d, x.abs().t() @ d.abs(), cap, torch.float32)).all()), e


# bf16 tiles of 128, 160 and 192 rows by 256 columns (and, in the first and the seventh, of 128 x 128): rows that end on such a tile, one before and one behind, of one row and none;
# columns around a multiple of 256, reductions of an odd and an even number of k-tiles with 8 k in the last one, of two k-tiles; no row counts
@pytest.mark.parametrize("cap,n,k,hint,counts", [(400, 2040, 136, 290, [256, 257, 255, 0, 1, 128, 384, 400]), (160, 4000, 520, 120, [128, 129, 127, 160, 1, 0, 64, 33]),
                                                 (620, 2056, 200, 490, [480, 481, 479, 620, 0, 1, 160, 161]), (620, 2048, 520, 500, [320, 640, 159, 97, 96, 95, 64, 65]),
                                                 (1100, 1032, 520, 1000, [960, 961, 959, 1100, 1, 192, 193, 97]), (2500, 2048, 72, 2000, [1920, 1921, 1919, 2500, 0, 1, 288, 289]),
                                                 (768, 1000, 520, 0, [768] * 8), (384, 4088, 200, 0, [384] * 8)])
def test_expert_gemm_low_tiles(cap, n, k, hint, counts):
    from planmoe_amd import ops
    print("case", cap, n, k, hint, flush=True)
    B, dtype = 8, torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(cap + n)
    a, w = torch.randn(B, cap, k, device=DEV, generator=g).to(dtype), torch.randn(B, k, n, device=DEV, generator=g).to(dtype)
    bias, h = torch.randn(B, n, device=DEV, generator=g).to(dtype), torch.randn(B, cap, n, device=DEV, generator=g).clamp(min=0).to(dtype)
    rows = [min(cap, c) for c in counts]
    for e, r in enumerate(rows):
        a[e, r:] = float("nan")
    wt, live = w.transpose(1, 2).contiguous(), torch.tensor([counts], dtype=torch.int32, device=DEV) if hint else None
    nn = torch.full((B, cap, n), 7.0, dtype=dtype, device=DEV)
    nt, masked = nn.clone(), nn.clone()
    kw = dict(live=live, rows_hint=hint)
    ops.expert_gemm("nn", a, w, bias, relu=True, out=nn, **kw)
    ops.expert_gemm("nt", a, wt, out=nt, **kw)
    _, db = ops.expert_gemm_relu_bwd(a, wt, h, out=masked, **kw)
    torch.cuda.synchronize()
    for e, r in enumerate(rows):
        ref, mag = a[e, :r].double() @ w[e].double(), a[e, :r].double().abs() @ w[e].double().abs()
        tol, biased = _bound(ref, mag, k, dtype), ref + bias[e].double()
        assert bool(((nn[e, :r].double() - biased.clamp(min=0)).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, dtype)).all()), e
        assert bool(((nt[e, :r].double() - ref).abs() <= tol).all()), e
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all()), e
        for out in (nn, nt, masked):
            assert bool((out[e, r:] == 7.0).all()), e
        stored = masked[e, :r].double()
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), max(r, 1), dtype)).all()), e


# Few rows where there are more pieces of 64 columns than compute units: up to 16 rows in 96 (nt) or 128 columns, up to 32 where those have a
# compute unit each, in tiles otherwise; columns that no width divides, an expert without rows, and one with all.
@pytest.mark.parametrize("B,n,k", [(8, 2568, 72), (16, 2488, 136), (7, 4104, 520), (64, 264, 1032)])
@pytest.mark.parametrize("m", [3, 16, 17, 32, 33, 64, 65])
def test_expert_gemm_few_rows_and_many_columns(B, n, k, m):
    from planmoe_amd import ops
    print("case", B, n, k, m, flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    dtype = torch.bfloat16
    live = torch.randint(0, m + 1, (1, B), generator=g, dtype=torch.int32)
    live[0, 0], live[0, 1] = 0, m
    a, bias = torch.randn(B, m, k, generator=g).to(dtype).to(DEV), torch.randn(B, n, generator=g).to(dtype).to(DEV)
    w, h = torch.randn(B, k, n, generator=g).to(dtype).to(DEV), torch.randn(B, m, n, generator=g).clamp(min=0).to(dtype).to(DEV)
    for e in range(B):
        a[e, int(live[0, e]):] = float("nan")
    wt = w.transpose(1, 2).contiguous()
    nn = torch.full((B, m, n), 7.0, dtype=dtype, device=DEV)
    nt, masked = nn.clone(), nn.clone()
    kw = dict(live=live.to(DEV), rows_hint=(m + 1) // 2)
    ops.expert_gemm("nn", a, w, bias, relu=True, out=nn, **kw)
    ops.expert_gemm("nt", a, wt, out=nt, **kw)
    _, db = ops.expert_gemm_relu_bwd(a, wt, h, out=masked, **kw)
    torch.cuda.synchronize()
    for e in range(B):
        r = int(live[0, e])
        x, y = a[e, :r].double(), w[e].double()
        ref, mag = x @ y, x.abs() @ y.abs()
        tol = _bound(ref, mag, k, dtype)
        biased = ref + bias[e].double()
        assert bool(((nn[e, :r].double() - biased.clamp(min=0)).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, dtype)).all())
        assert bool(((nt[e, :r].double() - ref).abs() <= tol).all())
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all())
        for out in (nn, nt, masked):
            assert bool((out[e, r:] == 7.0).all())
        stored = masked[e, :r].double()          # the sums are of what was stored
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), r, dtype)).all())


# Tiles of 64 x 64 with four k-tiles in LDS: one, two and three k-tiles more than a round of them, a piece of one; a k that is the slow index of one or
# both operands, rows in use below the capacity and none, NaN behind them; against the same product with the rows expected that take other tiles
# only by the rounding of its sums, and bit for bit against waves on their own where no split serves (n below 256).
@pytest.mark.parametrize("B,cap,n,k", [(3, 70, 68, 228), (4, 130, 260, 256), (2, 100, 520, 292), (5, 40, 132, 324), (3, 200, 300, 1028), (2, 257, 64, 384)])
def test_expert_gemm_fp32_four_stages(B, cap, n, k):
    from planmoe_amd import ops
    print("case", B, cap, n, k, flush=True)
    g = torch.Generator().manual_seed(cap + n + k)
    live = torch.tensor([[cap - 3, 0, 33, 1, 64][:B]], dtype=torch.int32)
    a, w = torch.randn(B, cap, k, generator=g), torch.randn(B, k, n, generator=g)
    h, bias = torch.randn(B, cap, n, generator=g).clamp(min=0), torch.randn(B, n, generator=g)
    for e in range(B):
        a[e, int(live[0, e]):] = float("nan")
    wt = w.transpose(1, 2).contiguous()
    a, w, wt, h, bias = (t.to(DEV) for t in (a, w, wt, h, bias))
    kw = dict(live=live.to(DEV), rows_hint=33)
    nn = torch.full((B, cap, n), 7.0, device=DEV)
    nt, masked = nn.clone(), nn.clone()
    ops.expert_gemm("nn", a, w, bias, relu=True, out=nn, **kw)
    ops.expert_gemm("nt", a, wt, out=nt, **kw)
    _, db = ops.expert_gemm_relu_bwd(a, wt, h, out=masked, **kw)
    # a^T b over the rows in use, whose number has to reach eight k-tiles: the operands' other way round
    rows = torch.tensor([[k - 5, 0, k, 226, 33][:B]], dtype=torch.int32)
    x, d = torch.randn(B, k, 72, generator=g), torch.randn(B, k, n, generator=g)
    for e in range(B):
        x[e, int(rows[0, e]):] = d[e, int(rows[0, e]):] = float("nan")
    tn = ops.expert_gemm("tn", x.to(DEV), d.to(DEV), live=rows.to(DEV), rows_hint=k)
    if n < 256:
        one = torch.empty_like(nn)
        ops.expert_gemm("nn", a, w, bias, relu=True, out=one, live=live.to(DEV), rows_hint=1)
    torch.cuda.synchronize()
    for e in range(B):
        r, q = int(live[0, e]), int(rows[0, e])
        y, z = a[e, :r].double(), w[e].double()
        ref, mag = y @ z, y.abs() @ z.abs()
        tol = _bound(ref, mag, k, torch.float32)
        assert bool(((nn[e, :r].double() - (ref + bias[e].double()).clamp(min=0)).abs() <= tol + _bound(ref, bias[e].double().abs()[None] + ref.abs(), 1, torch.float32)).all())
        assert bool(((nt[e, :r].double() - ref).abs() <= tol).all())
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all())
        for out in (nn, nt, masked):
            assert bool((out[e, r:] == 7.0).all())
        stored = masked[e, :r].double()          # the sums are of what was stored
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), r, torch.float32)).all())
        xs, ds = x[e, :q].double(), d[e, :q].double()
        assert bool(((tn[e].double().cpu() - xs.t() @ ds).abs() <= _bound(xs.t() @ ds, xs.abs().t() @ ds.abs(), k, torch.float32)).all())
        if n < 256: assert torch.equal(one[e, :r], nn[e, :r])


# Tiles of 128 x 128 with a compute unit each, four k-tiles of 64 in LDS: reductions of less than one, of one, of four, one more and pieces; rows in use of
# none, one, either side of half a tile and of a tile; columns of a piece; every form, the masked one's column sums.
@pytest.mark.parametrize("k", [8, 56, 64, 72, 256, 264, 520])
@pytest.mark.parametrize("cap,n,counts", [(66, 136, [66, 0, 33, 1, 65]), (300, 264, [0, 127, 128, 129, 300]), (257, 8, [257, 256, 255, 64, 63])])
def test_expert_gemm_tile_alone(cap, n, counts, k):
    from planmoe_amd import ops
    print("case", cap, n, counts, k, flush=True)
    g = torch.Generator().manual_seed(cap + n + k)
    B, dtype = 5, torch.bfloat16
    live = torch.tensor([counts], dtype=torch.int32)
    a, w = torch.randn(B, cap, k, generator=g).to(dtype), torch.randn(B, k, n, generator=g).to(dtype)
    h, bias, d = torch.randn(B, cap, n, generator=g).clamp(min=0).to(dtype), torch.randn(B, n, generator=g).to(dtype), torch.randn(B, cap, n, generator=g).to(dtype)
    for e in range(B):
        a[e, counts[e]:] = d[e, counts[e]:] = float("nan")
    a, w, h, bias, d = (t.to(DEV) for t in (a, w, h, bias, d))
    wt = w.transpose(1, 2).contiguous()
    nn = torch.full((B, cap, n), 7.0, dtype=dtype, device=DEV)
    nt, masked = nn.clone(), nn.clone()
    kw = dict(live=live.to(DEV), rows_hint=100)
    ops.expert_gemm("nn", a, w, bias, relu=True, out=nn, **kw)
    ops.expert_gemm("nt", a, wt, out=nt, **kw)
    _, db = ops.expert_gemm_relu_bwd(a, wt, h, out=masked, **kw)
    tn = ops.expert_gemm("tn", a, d, **kw)
    torch.cuda.synchronize()
    for e in range(B):
        r = counts[e]
        x, y = a[e, :r].double(), w[e].double()
        ref, mag = x @ y, x.abs() @ y.abs()
        tol = _bound(ref, mag, k, dtype)
        biased = ref + bias[e].double()
        assert bool(((nn[e, :r].double() - biased.clamp(min=0)).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, dtype)).all())
        assert bool(((nt[e, :r].double() - ref).abs() <= tol).all())
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all())
        for out in (nn, nt, masked):
            assert bool((out[e, r:] == 7.0).all())
        stored = masked[e, :r].double()          # the sums are of what was stored
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), r, dtype)).all())
        z = d[e, :r].double()
        assert bool(((tn[e].double() - x.t() @ z).abs() <= _bound(x.t() @ z, x.abs().t() @ z.abs(), cap, dtype)).all())


# fp32: the order of the sums is the buffer's shape's, not that of the rows in use or expected: a product over the rows in use (the layer as one
# node) has the bits of the one over the whole buffer (its steps).  Few rows expected of a capacity that is computed in parts and of one that is
# not, capacities of 80 and one piece more, rows for which the other way would be the faster one; a tn product's reduction over few rows and all
@pytest.mark.parametrize("B,cap,n,k,hint", [(16, 76, 1036, 1028, 60), (16, 100, 1036, 1028, 60), (16, 128, 2048, 512, 8), (8, 320, 1024, 1024, 100), (8, 200, 520, 512, 16),
                                            (16, 80, 1024, 512, 64), (16, 84, 2048, 512, 64), (8, 952, 320, 1120, 634), (4, 600, 512, 1024, 256), (4, 300, 1024, 1028, 200)])
def test_expert_gemm_fp32_does_not_depend_on_the_rows_in_use(B, cap, n, k, hint):
    from planmoe_amd import ops
    print("case", B, cap, n, k, hint, flush=True)
    g = torch.Generator(device=DEV).manual_seed(cap + n + k)
    counts = [min(cap, max(0, hint + 7 * (e % 5 - 2))) for e in range(B)]
    counts[0], counts[1] = 0, cap
    live = torch.tensor([counts], dtype=torch.int32, device=DEV)
    a, d = torch.randn(B, cap, k, device=DEV, generator=g), torch.randn(B, cap, n, device=DEV, generator=g)
    w, bias, h = torch.randn(B, k, n, device=DEV, generator=g), torch.randn(B, n, device=DEV, generator=g), torch.randn(B, cap, n, device=DEV, generator=g).clamp(min=0)
    for e, r in enumerate(counts):
        a[e, r:] = d[e, r:] = 0.0
    wt, kw = w.transpose(1, 2).contiguous(), dict(live=live, rows_hint=hint)
    for relu in (False, True):
        got, want = ops.expert_gemm("nn", a, w, bias, relu=relu, **kw), ops.expert_gemm("nn", a, w, bias, relu=relu)
        for e, r in enumerate(counts):
            assert torch.equal(got[e, :r], want[e, :r]), ("nn", relu, e)
    got, want = ops.expert_gemm("nt", a, wt, **kw), ops.expert_gemm("nt", a, wt)
    masked, _ = ops.expert_gemm_relu_bwd(a, wt, h, **kw)
    for e, r in enumerate(counts):
        assert torch.equal(got[e, :r], want[e, :r]), ("nt", e)
        assert torch.equal(masked[e, :r], torch.where(h[e, :r] > 0, want[e, :r], torch.zeros((), device=DEV))), ("masked", e)
    got, want = ops.expert_gemm("tn", a, d, **kw), ops.expert_gemm("tn", a, d)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


# A NaN goes through the relu whatever its sign, from an operand and from the bias, in every kernel: few rows on waves, a tile alone, tiles of 128 and 256
# rows by 256 columns and 128 x 128, and in fp32
@pytest.mark.parametrize("dtype,B,m,n,k", [(torch.bfloat16, 2, 16, 72, 64), (torch.bfloat16, 2, 40, 72, 64), (torch.bfloat16, 8, 500, 2048, 200), (torch.bfloat16, 8, 4096, 1024, 64),
                                           (torch.bfloat16, 8, 1030, 1032, 72), (torch.float32, 2, 16, 72, 64), (torch.float32, 2, 100, 72, 64)])
def test_expert_gemm_relu_keeps_nan_of_either_sign(dtype, B, m, n, k):
    from planmoe_amd import ops
    print("case", dtype, B, m, n, k, flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n)
    a, w = torch.randn(B, m, k, device=DEV, generator=g).to(dtype), torch.randn(B, k, n, device=DEV, generator=g).to(dtype)
    bias = torch.randn(B, n, device=DEV, generator=g).to(dtype)
    bits, sign = (torch.int16, -64) if dtype == torch.bfloat16 else (torch.int32, -4194304)        # 0xffc0 (0000): a NaN with its sign set
    bias.view(bits)[0, 3] = sign
    bias[0, 6], bias[1, 5] = float("nan"), float("-inf")
    if dtype == torch.bfloat16: bias.view(bits)[1, 8:10] = torch.tensor([-1, -127], dtype=bits, device=DEV)
    a.view(bits)[B - 1, m - 1, 2] = sign
    got = ops.expert_gemm("nn", a, w, bias, relu=True)
    want = torch.relu(torch.bmm(a.float(), w.float()) + bias.float()[:, None])
    torch.cuda.synchronize()
    assert torch.equal(got.isnan(), want.isnan()) and bool((got[1, :m - 1, 5] == 0).all()) and bool((got[~got.isnan()] >= 0).all())


# Every kernel of the experts' products by its name, and each form that it has: nn, nt and the masked nt with its column sums ("rows"), a^T b ("tn").  Rows in
# use of none, one, either side of the tiles' sides, a capacity's and the rest as expected, NaN behind them and a sentinel in what must not be
# written; an even and an odd number of k-tiles, each with a piece of one; columns that no tile divides.  What the shapes are for is asserted: the
# rules between the kernels are fitted to times and move.
IN_KERNEL = [
    (torch.bfloat16, "rows", "few rows", 4, 8, 16, 200, 6), (torch.bfloat16, "rows", "128x128 alone", 4, 300, 264, 136, 200),
    (torch.bfloat16, "rows", "128x128", 5, 2734, 160, 200, 2734), (torch.bfloat16, "rows", "128x128", 8, 1697, 144, 144, 1697),
    (torch.bfloat16, "rows", "128x256", 8, 2618, 144, 720, 2356), (torch.bfloat16, "rows", "128x256", 8, 139, 3832, 440, 125),
    (torch.bfloat16, "rows", "160x256", 8, 801, 1160, 200, 801), (torch.bfloat16, "rows", "160x256", 8, 2118, 392, 136, 2118),
    (torch.bfloat16, "rows", "192x256", 5, 2722, 520, 200, 2722), (torch.bfloat16, "rows", "192x256", 8, 2765, 280, 144, 2765),
    (torch.bfloat16, "rows", "256x256", 8, 429, 2608, 200, 429), (torch.bfloat16, "rows", "256x256", 8, 1551, 792, 136, 1551),
    (torch.bfloat16, "rows", "256x256 and quarters", 8, 1755, 2528, 1264, 1755), (torch.bfloat16, "rows", "256x256 and quarters", 8, 2013, 2160, 1584, 2013),
    (torch.bfloat16, "tn", "128x128 alone", 4, 203, 16, 136, 182), (torch.bfloat16, "tn", "128x128 alone", 4, 260, 264, 1144, 234),
    (torch.bfloat16, "tn", "128x128", 8, 202, 136, 1544, 202), (torch.bfloat16, "tn", "128x128", 8, 267, 144, 1552, 240),
    (torch.bfloat16, "tn", "256x256", 8, 201, 2072, 392, 160), (torch.bfloat16, "tn", "256x256", 8, 270, 2712, 264, 216),
    (torch.bfloat16, "tn", "256x256 and quarters", 4, 1098, 2784, 1512, 1098), (torch.bfloat16, "tn", "256x256 and quarters", 4, 1288, 2480, 1576, 1288),
    (torch.float32, "rows", "f32 waves", 4, 9, 16, 168, 8), (torch.float32, "rows", "f32 64x64", 4, 37, 16, 164, 37),
    (torch.float32, "rows", "f32 64x64 four stages", 16, 81, 880, 264, 79), (torch.float32, "rows", "f32 64x64 four stages", 16, 81, 844, 240, 79),
    (torch.float32, "rows", "f32 32x32", 8, 70, 548, 260, 70), (torch.float32, "rows", "f32 32x32", 8, 44, 780, 240, 43),
    (torch.float32, "rows", "f32 32x32 eight stages", 4, 70, 68, 268, 60), (torch.float32, "rows", "f32 32x32 eight stages", 4, 78, 36, 236, 70),
    (torch.float32, "rows", "f32 128x128", 8, 73, 3232, 176, 65),
    (torch.float32, "rows", "f32 parts 64x64", 4, 2618, 260, 292, 2356), (torch.float32, "rows", "f32 parts 64x64", 8, 324, 1052, 260, 291),
    (torch.float32, "rows", "f32 parts 128x128", 8, 389, 848, 300, 311), (torch.float32, "rows", "f32 parts 128x128", 4, 388, 1736, 268, 349),
    (torch.float32, "rows", "f32 parts 256x128", 5, 2382, 388, 292, 2382), (torch.float32, "rows", "f32 parts 256x128", 16, 512, 1024, 1024, 512),
    (torch.float32, "tn", "f32 64x64", 4, 240, 16, 136, 192), (torch.float32, "tn", "f32 64x64 four stages", 4, 266, 16, 144, 239),
    (torch.float32, "tn", "f32 128x128", 5, 255, 2472, 196, 204), (torch.float32, "tn", "f32 parts 64x64", 8, 247, 392, 260, 247),
    (torch.float32, "tn", "f32 parts 128x128", 4, 225, 264, 1732, 180), (torch.float32, "tn", "f32 parts 128x128", 8, 200, 652, 332, 160),
    (torch.float32, "tn", "f32 parts 256x128", 8, 227, 1468, 388, 227), (torch.float32, "tn", "f32 parts 256x128", 4, 203, 3404, 332, 203)]


@pytest.mark.parametrize("dtype,form,kernel,B,cap,n,k,hint", IN_KERNEL)
def test_expert_gemm_in_every_kernel(dtype, form, kernel, B, cap, n, k, hint):
    from planmoe_amd import ops
    print("case", dtype, form, kernel, B, cap, n, k, hint, flush=True)
    relu = dtype == torch.bfloat16 or "parts" not in kernel          # (a relu keeps the fp32 matrix cores' order of sums)
    if form == "tn":
        assert ops.expert_gemm_kernel("tn", dtype, B, k, n, cap, counted=True, rows_hint=hint) == kernel
    else:
        assert ops.expert_gemm_kernel("nn", dtype, B, cap, n, k, relu=relu, counted=True, rows_hint=hint) == kernel
        assert ops.expert_gemm_kernel("nt", dtype, B, cap, n, k, counted=True, rows_hint=hint) == kernel
    g = torch.Generator(device=DEV).manual_seed(cap + n + k)
    edges = [cap, 0, 1, hint, 129, 256, 65, 127, 63, 257, 192, 160, 193, 161, 64, 128]
    if form == "rows" and "quarters" in kernel:
        edges = [hint] * 4 + [0, 1, 129, 257]       # (a round of 256 tiles, and a quarter of one)
    rows = [min(cap, edges[e]) for e in range(B)]
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g).to(dtype)
    live, a = torch.tensor([rows], dtype=torch.int32, device=DEV), rand(B, cap, k)
    for e, r in enumerate(rows):
        a[e, r:] = float("nan")
    kw = dict(live=live, rows_hint=hint)
    if form == "tn":
        dy = rand(B, cap, n)
        for e, r in enumerate(rows):
            dy[e, r:] = float("nan")
        got = ops.expert_gemm("tn", a, dy, **kw)
        torch.cuda.synchronize()
        for e, r in enumerate(rows):
            x, d = a[e, :r].double().t().contiguous(), dy[e, :r].double()
            ref = x @ d
            assert bool(((got[e].double() - ref).abs() <= _bound(ref, x.abs() @ d.abs(), cap, dtype)).all()), (e, r)
        return
    w, bias, h = rand(B, k, n), rand(B, n), rand(B, cap, n).clamp(min=0)
    wt = w.transpose(1, 2).contiguous()
    nn = torch.full((B, cap, n), 7.0, dtype=dtype, device=DEV)
    nt, masked = nn.clone(), nn.clone()
    ops.expert_gemm("nn", a, w, bias, relu=relu, out=nn, **kw)
    ops.expert_gemm("nt", a, wt, out=nt, **kw)
    _, db = ops.expert_gemm_relu_bwd(a, wt, h, out=masked, **kw)
    torch.cuda.synchronize()
    for e, r in enumerate(rows):
        x, y = a[e, :r].double(), w[e].double()
        ref, mag = x @ y, x.abs() @ y.abs()
        tol, biased = _bound(ref, mag, k, dtype), ref + bias[e].double()
        assert bool(((nn[e, :r].double() - (biased.clamp(min=0) if relu else biased)).abs() <= tol + _bound(biased, bias[e].double().abs()[None], 1, dtype)).all()), (e, r)
        assert bool(((nt[e, :r].double() - ref).abs() <= tol).all()), (e, r)
        assert bool(((masked[e, :r].double() - ref * (h[e, :r] > 0)).abs() <= tol).all()), (e, r)
        for out in (nn, nt, masked):
            assert bool((out[e, r:] == 7.0).all()), (e, r)
        stored = masked[e, :r].double()          # the sums are of what was stored
        assert bool(((db[e].double() - stored.sum(0)).abs() <= _bound(stored.sum(0), stored.abs().sum(0), max(r, 1), dtype)).all()), (e, r)


# The tile alone in 128 columns, where 64 would be more work-groups than there are compute units (the shapes above and test_expert_gemm_tile_alone's are
# in 64): reductions of three k-tiles, of one more than LDS holds and of many
@pytest.mark.parametrize("form,B,cap,n,k,hint", [("rows", 8, 128, 2056, 136, 110), ("rows", 8, 128, 2056, 328, 110), ("rows", 4, 128, 4104, 1032, 100), ("tn", 4, 260, 1208, 392, 234),
                                                 ("tn", 4, 600, 1208, 392, 600)])
def test_expert_gemm_tile_alone_in_128_columns(form, B, cap, n, k, hint):
    units = torch.cuda.get_device_properties(0).multi_processor_count
    narrow = B * ((n + 63) // 64) * (1 if form == "rows" else (k + 127) // 128)          # (both widths have one name)
    assert narrow > (units if form == "rows" else 0.8 * units)
    test_expert_gemm_in_every_kernel(torch.bfloat16, form, "128x128 alone", B, cap, n, k, hint)


# The parts are no less precise than the fp32 matrix cores (which serve the same product under a relu: where a result is positive, that is the product):
# the results and their sums over the rows, in which what is rounded one way adds up, for operands of both signs, behind a relu, and positive
@pytest.mark.parametrize("form,kernel,B,m,n,k", [("nn", "f32 parts 256x128", 16, 512, 1024, 1024), ("nt", "f32 parts 256x128", 16, 512, 1024, 1024),
                                                 ("tn", "f32 parts 256x128", 16, 1024, 1024, 512), ("nn", "f32 parts 128x128", 8, 1024, 512, 512),
                                                 ("tn", "f32 parts 128x128", 8, 332, 652, 200), ("nt", "f32 parts 64x64", 8, 750, 1536, 768),
                                                 ("nn", "f32 parts 64x64", 8, 300, 2048, 2048), ("nn", "f32 parts 256x128", 2, 4096, 2048, 4096)])
@pytest.mark.parametrize("operands", ["normal", "relu", "positive"])
def test_expert_gemm_fp32_in_parts_is_no_less_precise(form, kernel, B, m, n, k, operands):
    from planmoe_amd import ops
    print("case", form, kernel, B, m, n, k, operands, flush=True)
    assert ops.expert_gemm_kernel(form, torch.float32, B, m, n, k) == kernel
    assert "parts" not in ops.expert_gemm_kernel(form, torch.float32, B, m, n, k, relu=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = torch.randn(*((B, k, m) if form == "tn" else (B, m, k)), device=DEV, generator=g)
    b = torch.randn(*((B, n, k) if form == "nt" else (B, k, n)), device=DEV, generator=g)
    a, b = (a.clamp(min=0), b) if operands == "relu" else (a.abs(), b.abs()) if operands == "positive" else (a, b)
    got, fp32, ref = ops.expert_gemm(form, a, b).double(), ops.expert_gemm(form, a, b, relu=True).double(), _fp64(form, a, b)[0]
    torch.cuda.synchronize()
    there = (fp32 > 0) & (got > 0) & (ref > 0)
    parts, whole = (got - ref) * there, (fp32 - ref) * there
    assert float(parts.norm()) <= float(whole.norm())
    assert float(parts.sum(1).norm()) <= float(whole.sum(1).norm())


@pytest.mark.parametrize("shares", [2, 5, 8, 9, 16])
def test_sums_of_shares_are_added_in_pairs(shares):
    """Shares of 32 rows: the first one's sum is 1, those of the others half a unit of its last place, which one after the other are lost.  Eight in
    pairs have three roundings, a wave's sums up to four more."""
    from planmoe_amd import ops
    from planmoe_amd._lib import check, lib
    a = torch.zeros(1, 32 * shares, 64, device=DEV)
    a[0, ::32] = 2.0 ** -24
    a[0, 0] = 1.0
    out = torch.empty(1, 64, device=DEV)
    ws = torch.empty(lib.planmoe_rows_colsum_workspace_bytes(1, 32 * shares, 64), dtype=torch.uint8, device=DEV)
    check(lib.planmoe_rows_colsum(ops._ptr(a), ops._dt(a, "t"), 1, 32 * shares, 64, None, 1, 1, ops._ptr(out), ops._ptr(ws), ws.numel(), ops._stream(a)))
    torch.cuda.synchronize()
    want = 1.0 + (shares - 1) * 2.0 ** -24
    assert bool(((out.double() - want).abs() <= 2.0 ** -23).all()), (out[0, 0].item() - 1.0) * 2 ** 24


# fp32, waves on their own: 16 and 32 rows, 16, 32 and 64 columns, work-groups of one and four waves, past the caches; columns and reductions that
# nothing divides.  The same rows in a larger buffer go through the tiles, and the sums have the same order.
@pytest.mark.parametrize("form,B,cap,n,k", [
    ("nn", 4, 12, 52, 200), ("nn", 16, 16, 520, 36), ("nn", 16, 8, 1036, 148), ("nn", 16, 9, 1300, 20), ("nn", 16, 4, 2100, 2080),
    ("nn", 4, 40, 52, 200), ("nn", 16, 33, 1060, 44), ("nn", 16, 20, 1700, 300),
    ("nt", 4, 12, 52, 200), ("nt", 16, 16, 1036, 148), ("nt", 4, 40, 68, 200), ("nt", 16, 33, 1060, 44), ("nt", 16, 14, 572, 1172), ("nt", 16, 4, 1020, 260)])
def test_expert_gemm_few_fp32_rows_have_the_tiles_bits(form, B, cap, n, k):
    from planmoe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n + k)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    hint, more = min(cap, 30), 100
    assert ops.expert_gemm_kernel(form, torch.float32, B, cap, n, k, relu=form == "nn", counted=True, rows_hint=hint) == "f32 waves"
    edges = [cap, 0, 1, hint, 16, 17, 31, 33, 15, 32, 2, 5]
    rows = [min(cap, edges[e % 12]) for e in range(B)]
    live = torch.tensor([rows], dtype=torch.int32, device=DEV)
    wide = rand(B, more, k)
    few, w, bias = wide[:, :cap].contiguous(), rand(B, k, n) if form == "nn" else rand(B, n, k), rand(B, n)
    for e, r in enumerate(rows):
        few[e, r:] = float("nan")
    sentinel = lambda rows: torch.full((B, rows, n), 7.0, device=DEV)
    kw = dict(live=live, relu=form == "nn")
    got = ops.expert_gemm(form, few, w, bias, out=sentinel(cap), rows_hint=hint, **kw)
    want = ops.expert_gemm(form, wide, w, bias, out=sentinel(more), rows_hint=more, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got, want[:, :cap])
    if form == "nt":
        h = rand(B, more, n)
        got, db = ops.expert_gemm_relu_bwd(few, w, h[:, :cap].contiguous(), live=live, out=sentinel(cap), rows_hint=hint)
        want, _ = ops.expert_gemm_relu_bwd(wide, w, h, live=live, out=sentinel(more), rows_hint=more)
        torch.cuda.synchronize()
        assert torch.equal(got, want[:, :cap])
        _column_sums_hold(db, got, rows, cap)


def _column_sums_hold(db, got, rows, cap):
    for e, r in enumerate(rows):
        ref = got[e, :r].double().sum(0)
        # (at most cap additions, each rounded to 2^-24 of the sum so far)
        assert bool(((db[e].double() - ref).abs() <= cap * 2.0 ** -24 * got[e, :r].double().abs().sum(0)).all())


# fp32 tiles of 32 x 32, five and eight k-tiles in LDS, and of 64 x 64 with small ones of 16 and 32 rows behind them; columns, reductions
# and row counts around their sides, with and without counts.  Each 32 rows go through the waves as well, among more columns, and the bits are theirs.
@pytest.mark.parametrize("counted", [True, False])
@pytest.mark.parametrize("kernel,form,B,cap,n,k,hint", [
    ("f32 32x32 eight stages", "nn", 4, 12, 52, 300, 9), ("f32 32x32", "nn", 16, 20, 1036, 292, 20), ("f32 32x32 eight stages", "nn", 2, 70, 148, 724, 70),
    ("f32 32x32", "nn", 8, 163, 260, 2044, 163), ("f32 32x32 eight stages", "nn", 1, 33, 4, 228, 33), ("f32 32x32 eight stages", "nt", 4, 40, 68, 236, 30),
    ("f32 32x32", "nt", 16, 33, 1060, 236, 30), ("f32 32x32 eight stages", "nt", 3, 97, 100, 240, 97), ("f32 64x64 four stages", "nn", 16, 108, 512, 1536, 97),
    ("f32 64x64 four stages", "nt", 16, 108, 1028, 252, 97), ("f32 64x64 four stages", "nn", 16, 81, 880, 264, 79), ("f32 64x64 four stages", "nt", 16, 81, 844, 252, 79), ("f32 64x64 four stages", "nt", 16, 81, 880, 264, 79)])
def test_expert_gemm_small_fp32_tiles_have_the_waves_bits(kernel, form, B, cap, n, k, hint, counted):
    from planmoe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n + k)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    assert ops.expert_gemm_kernel(form, torch.float32, B, cap, n, k, relu=form == "nn", counted=counted, rows_hint=hint) == kernel
    edges = [cap, 0, 1, 65, 80, 81, 96, 97, 15, 16, 17, 31, 32, 33, 63, 64]
    rows = [min(cap, edges[e % 16]) if counted else cap for e in range(B)]
    live = torch.tensor([rows], dtype=torch.int32, device=DEV) if counted else None
    a, w, bias, h = rand(B, cap, k), rand(B, k, n), rand(B, n), rand(B, cap, n)
    if not counted and form == "nt":
        a[0, 0, k - 1], w[0, k - 1, 1] = float("inf"), float("nan")
    columns = -(-25600 // B // 4) * 4
    many = w.repeat(1, 1, -(-columns // n))[:, :, :columns].contiguous()
    assert columns >= n and ops.expert_gemm_kernel("nn", torch.float32, B, 32, columns, k) == "f32 waves"
    want = torch.cat([ops.expert_gemm("nn", a[:, i:i + 32].contiguous(), many)[:, :, :n] for i in range(0, cap, 32)], 1)
    for e, r in enumerate(rows):
        a[e, r:] = float("nan")
    b = w if form == "nn" else w.transpose(1, 2).contiguous()
    sentinel = torch.full((B, cap, n), 7.0, device=DEV)
    got = ops.expert_gemm(form, a, b, bias, relu=form == "nn", live=live, rows_hint=hint, out=sentinel.clone())
    ref = want + bias[:, None]
    if form == "nn":
        ref = torch.where(ref < 0, torch.zeros_like(ref), ref)
    there = (torch.arange(cap, device=DEV)[None, :] < torch.tensor(rows, device=DEV)[:, None])[:, :, None]
    same = lambda x, y: torch.equal(torch.where(there, y, sentinel).nan_to_num(123.0), x.nan_to_num(123.0))
    assert same(got, ref)
    if form == "nt":
        got, db = ops.expert_gemm_relu_bwd(a, b, h, live=live, rows_hint=hint, out=sentinel.clone())
        assert same(got, torch.where(h > 0, want, torch.zeros_like(want)))
        if counted:
            _column_sums_hold(db, got, rows, cap)


# A row an expert, of which any number may be without one: tiles of 64 x 64, none of them whole, where waves would do for all; the bits are the waves'
@pytest.mark.parametrize("B,cap,n,k", [(16, 4, 1700, 300), (8, 12, 3300, 260)])
@pytest.mark.parametrize("rows", [[0, 0, 1], [1], [0], [4, 0, 2, 0, 0, 1, 12]])
def test_expert_gemm_of_a_row_an_expert(B, cap, n, k, rows):
    from planmoe_amd import ops
    assert [ops.expert_gemm_kernel("nn", torch.float32, B, cap, n, k, counted=True, relu=True, rows_hint=h) for h in (1, 2)] == ["f32 64x64 four stages", "f32 waves"]
    g = torch.Generator(device=DEV).manual_seed(n)
    rows = [min(cap, rows[e % len(rows)]) for e in range(B)]
    live = torch.tensor([rows], dtype=torch.int32, device=DEV)
    a, w, bias = (torch.randn(*shape, device=DEV, generator=g) for shape in ((B, cap, k), (B, k, n), (B, n)))
    for e, r in enumerate(rows):
        a[e, r:] = float("nan")
    got, want = (ops.expert_gemm("nn", a, w, bias, relu=True, live=live, rows_hint=h, out=torch.full((B, cap, n), 7.0, device=DEV)) for h in (1, 2))
    assert torch.equal(got, want) and all(bool((got[e, r:] == 7.0).all() and got[e, :r].isfinite().all()) for e, r in enumerate(rows))


# fp32 tiles of 64 x 64 where those of 32 x 32 are several a compute unit in turn and measured slower (16.7 and 18.9 us the first), and the other way round
@pytest.mark.parametrize("kernel,form,B,cap,n,k,hint", [
    ("f32 64x64 four stages", "nn", 4, 320, 1024, 512, 256), ("f32 64x64 four stages", "nt", 4, 320, 1024, 512, 256), ("f32 32x32", "nn", 4, 320, 512, 1024, 256),
    ("f32 64x64 four stages", "nn", 8, 35, 1976, 384, 35), ("f32 64x64 four stages", "nn", 4, 114, 1792, 388, 114), ("f32 32x32", "nt", 4, 95, 2104, 2848, 95),
    ("f32 32x32", "nt", 8, 197, 1024, 3520, 157), ("f32 waves", "nt", 8, 5, 1408, 384, 3), ("f32 waves", "nt", 4, 4, 3784, 228, 4),
    ("f32 64x64 four stages", "nn", 16, 4, 3712, 2328, 1), ("f32 64x64 four stages", "nn", 8, 4, 4096, 512, 1), ("f32 waves", "nn", 8, 4, 4096, 512, 2),
    ("f32 waves", "nn", 8, 4, 4096, 200, 1), ("f32 32x32", "nt", 4, 15, 3636, 1920, 15), ("f32 32x32 eight stages", "nt", 16, 7, 448, 524, 5)])
def test_expert_gemm_fp32_tiles_by_what_they_measured(kernel, form, B, cap, n, k, hint):
    from planmoe_amd import ops
    assert ops.expert_gemm_kernel(form, torch.float32, B, cap, n, k, relu=form == "nn", counted=True, rows_hint=hint) == kernel


# Weight gradients over few rows, stored past the caches and plainly, 64, 128 and 256 columns of a wave; sizes that nothing divides.  The same rows in a
# larger buffer go through the tiles, and the sums have the same order.
@pytest.mark.parametrize("dtype,B,cap,m,n", [
    (torch.float32, 8, 1, 1028, 1024), (torch.float32, 8, 17, 1036, 1060), (torch.float32, 4, 100, 1024, 2084), (torch.float32, 8, 24, 2052, 4100),
    (torch.float32, 8, 150, 712, 1024), (torch.bfloat16, 4, 1, 8, 16), (torch.bfloat16, 4, 16, 40, 64), (torch.bfloat16, 8, 33, 264, 1032),
    (torch.bfloat16, 4, 90, 1032, 1024), (torch.bfloat16, 3, 12, 72, 2056), (torch.bfloat16, 3, 24, 200, 520)])
def test_expert_gemm_weight_gradients_of_few_rows_have_the_tiles_bits(dtype, B, cap, m, n):
    from planmoe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(m + n)
    hint, more = min(cap, 100 if dtype == torch.float32 else 60), 300
    assert ops.expert_gemm_kernel("tn", dtype, B, m, n, cap, counted=True, rows_hint=hint) == ("f32 parts few rows of a^T b" if dtype == torch.float32 else "few rows of a^T b")
    tiles = ops.expert_gemm_kernel("tn", dtype, B, m, n, more, counted=True, rows_hint=more)
    assert "few rows" not in tiles and (dtype != torch.float32 or "parts" in tiles)
    edges = [cap, 0, 1, hint, 16, 17, 31, 33]
    rows = [min(cap, edges[e % 8]) for e in range(B)]
    live = torch.tensor([rows], dtype=torch.int32, device=DEV)
    a, dy = (torch.randn(B, more, w, device=DEV, generator=g).to(dtype) for w in (m, n))
    a[B - 1, 0, 3], dy[0, 0, 5] = float("inf"), float("nan")
    few, few_dy = a[:, :cap].contiguous(), dy[:, :cap].contiguous()
    for e, r in enumerate(rows):
        few[e, r:], few_dy[e, r:] = float("nan"), float("nan")
    behind = torch.full((B * m * n + 64,), 7.0, dtype=dtype, device=DEV)
    out = behind[:B * m * n].view(B, m, n)
    got = ops.expert_gemm("tn", few, few_dy, live=live, rows_hint=hint, out=out)
    want = ops.expert_gemm("tn", a, dy, live=live, rows_hint=more)
    torch.cuda.synchronize()
    assert bool((behind[B * m * n:] == 7.0).all())
    assert torch.equal(got.isnan(), want.isnan())
    # (in parts a wave that meets what is not finite sums again in another order, and waves are not the same everywhere)
    whole = [e for e in range(B) if bool(want[e].isfinite().all())]
    assert len(whole) >= B - 2 and all(torch.equal(got[e], want[e]) for e in whole)
    for e in set(range(B)) - set(whole):
        keep = want[e].isfinite()
        assert torch.equal(got[e].isfinite(), keep)
        size = few[e, :rows[e]].double().abs().t().contiguous() @ few_dy[e, :rows[e]].double().abs()
        # (up to cap products rounded to 2^-24 and as many sums, twice; a bf16 result is rounded to 2^-8 on top)
        bound = (4 * cap * 2.0 ** -24 + (0 if dtype == torch.float32 else 2.0 ** -8)) * size
        assert bool(((got[e].double() - want[e].double()).abs() <= bound)[keep].all())
