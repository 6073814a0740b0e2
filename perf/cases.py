"""The work that a user has this framework do, as cases that can be timed and compared.

Five kinds, each through the public entry points:

  layer   moe_layer with its built-in expert FFN: "infer" is a forward pass without autograd (decode
          at a few tokens, prefill at many), "train" a forward and a backward pass
  route   the functional API: extract_critical, fast_encode, fast_decode, and their backward pass
  send    the send side kept as a plan (ForwardInt8Plan): gate, routing, dispatch, int8 codes
  bwd     the backward pass of the combine with the int8 codec on the gradient buffer, and that of
          the dispatch
  codec   a compressor on the all-to-all buffer: compress, hand-over, decompress
"""
import math

import torch

import planmoe_amd
from planmoe_amd import compressor, ops

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    layer = {"kind": "layer", "experts": 8, "top_k": 2, "factor": 1.25, "dtype": "bf16"}
    return [
        # one decode step of a small batch: every launch and all host work counts
        dict(layer, name="decode_8", mode="infer", tokens=8, dim=1024, hidden=4096, codec="no"),
        # a ragged prompt through the int8 all-to-all codec
        dict(layer, name="prefill_1999", mode="infer", tokens=1999, dim=2048, hidden=2048, codec="int8"),
        # a full prefill batch at the Mixtral-like size (16384 x 4096, 8 experts, top-2)
        dict(layer, name="prefill_16384", mode="infer", tokens=16384, dim=4096, hidden=4096, codec="int8"),
        # a small training step in fp32, no codec: what a first experiment or a test runs
        dict(layer, name="train_small_fp32", mode="train", tokens=512, dim=512, hidden=1024, experts=4, dtype="fp32", codec="no"),
        # the reference's own example: batch 8 x sequence 2048, model_dim 1024, capacity factor 1.2
        dict(layer, name="train_16384_int8", mode="train", tokens=16384, dim=1024, hidden=4096, factor=1.2, codec="int8"),
        # fp32 training with the lossy codec on both exchanges
        dict(layer, name="train_4096_zfp", mode="train", tokens=4096, dim=1024, hidden=1024, experts=16, factor=1.0, dtype="fp32",
             codec="zfp"),
        # routing and dispatch / combine by the functional API, forward and backward (8192 x 2048 fp32, 2 experts)
        {"name": "route_8192_fp32", "kind": "route", "tokens": 8192, "dim": 2048, "experts": 2, "top_k": 2, "factor": 1.0,
         "dtype": "fp32", "backward": True},
        # the same with nothing round: rows that no vector width divides, three choices, fp16
        {"name": "route_odd_fp16", "kind": "route", "tokens": 3001, "dim": 1030, "experts": 10, "top_k": 3, "factor": 1.1,
         "dtype": "fp16", "backward": True},
        # the send side of a serving loop at 16384 x 4096, 8 experts, top-2
        {"name": "send_16384", "kind": "send", "tokens": 16384, "dim": 4096, "experts": 8, "top_k": 2, "factor": 1.25, "skew": 0.0},
        # many experts, one choice, skewed routing that overflows the capacity (Zipf 1.2 on the logits)
        {"name": "send_64_experts", "kind": "send", "tokens": 32768, "dim": 2048, "experts": 64, "top_k": 1, "factor": 1.0, "skew": 1.2},
        # the fp32 buffer of 16 experts x 8192 slots x 1024 through the fixed-rate codec ...
        {"name": "codec_zfp", "kind": "codec", "codec": "zfp", "experts": 16, "slots": 8192, "dim": 1024, "empty": 0.0, "dtype": "fp32"},
        # ... and a smaller one with a third of its slots empty through the lossless codec
        {"name": "codec_lz", "kind": "codec", "codec": "lz", "experts": 16, "slots": 2048, "dim": 1024, "empty": 0.3, "dtype": "fp32"},
    ]


def _log(rng, low, high, step=1):
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "route", "send", "bwd", "codec"])
    factor = rng.choice([1.0, 1.1, 1.2, 1.25, 1.5])
    if kind == "layer":
        mode = rng.choice(["infer", "train"])
        codec = rng.choice(["no", "int8", "int8", "zfp", "lz"])
        dtype = "fp32" if codec in ("zfp", "lz") else rng.choice(["bf16", "bf16", "bf16", "fp32"])
        experts = rng.choice([4, 8, 8, 16])
        step = rng.choice([8, 64, 256])
        dim = _log(rng, 256, 4096, step)
        hidden = _log(rng, 256, 4096, step)
        most = 16384
        # a pass stays below the largest listed one: fp32 products run at a sixteenth of the bf16 rate, and a
        # backward pass is twice a forward pass
        while 4.0 * most * 2 * dim * hidden * factor * (3 if mode == "train" else 1) * (16 if dtype == "fp32" else 1) > 2.0e12:
            most //= 2
        return {"kind": kind, "mode": mode, "tokens": _log(rng, 1, most), "dim": dim, "hidden": hidden, "experts": experts,
                "top_k": rng.choice([1, 2, 2]), "factor": factor, "dtype": dtype, "codec": codec}
    if kind == "route":
        return {"kind": kind, "tokens": _log(rng, 16, 16384), "dim": _log(rng, 64, 4096, rng.choice([2, 8, 128])),
                "experts": _log(rng, 2, 64), "top_k": rng.choice([1, 2, 2]), "factor": factor,
                "dtype": rng.choice(["bf16", "fp16", "fp32"]), "backward": rng.random() < 0.6}
    if kind == "send":
        return {"kind": kind, "tokens": _log(rng, 32, 32768), "dim": _log(rng, 256, 4096, rng.choice([8, 256])),
                "experts": _log(rng, 4, 64), "top_k": rng.choice([1, 2, 2]), "factor": factor, "skew": rng.choice([0.0, 0.0, 1.2])}
    if kind == "bwd":
        return {"kind": kind, "tokens": _log(rng, 256, 16384), "dim": _log(rng, 256, 4096, rng.choice([8, 256])),
                "experts": _log(rng, 2, 16), "top_k": 2, "factor": factor, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    codec = rng.choice(["int8", "zfp", "lz"])
    return {"kind": kind, "codec": codec, "experts": rng.choice([4, 8, 16]), "slots": _log(rng, 16, 4096, 4),
            "dim": _log(rng, 256, 2048, rng.choice([4, 128])), "empty": rng.choice([0.0, 0.1, 0.3]),
            "dtype": rng.choice(["bf16", "fp32"]) if codec == "int8" else "fp32"}


def _randn(gen, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV) * scale).to(dtype)


def _capacity(case, alignment=4):
    k = min(case["top_k"], case["experts"])
    return ops.capacity(case["tokens"], case["experts"], k, case["factor"], alignment)


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    if kind == "layer":
        T, M, dtype = case["tokens"], case["dim"], DTYPES[case["dtype"]]
        torch.manual_seed(seed)
        with torch.device(DEV):
            layer = planmoe_amd.moe_layer({"type": "top", "k": case["top_k"], "capacity_factor": case["factor"], "fp32_gate": True},
                                          M, experts={"type": "ffn", "count_per_node": case["experts"],
                                                      "hidden_size_per_expert": case["hidden"]},
                                          compress_name=case["codec"])
        train = case["mode"] == "train"
        layer = layer.to(dtype).train(train)
        x = _randn(gen, T, M, dtype=dtype).requires_grad_(train)
        state = {"case": case, "layer": layer, "x": x}
        if train:
            state["grad"] = _randn(gen, T, M, dtype=dtype)       # what the layers above send back
            state["loss_weight"] = torch.full((), 0.01, device=DEV)
        return state
    if kind == "route":
        T, dtype = case["tokens"], DTYPES[case["dtype"]]
        scores = torch.softmax(_randn(gen, T, case["experts"]), 1)
        x = _randn(gen, T, case["dim"], dtype=dtype)
        state = {"case": case, "scores": scores, "x": x}
        if case["backward"]:
            scores.requires_grad_(True)
            x.requires_grad_(True)
            state["grad"] = _randn(gen, T, case["dim"], dtype=dtype)
        return state
    if kind == "send":
        T, M, E = case["tokens"], case["dim"], case["experts"]
        x = _randn(gen, T, M, dtype=torch.bfloat16)
        wg = _randn(gen, E, M, dtype=torch.bfloat16, scale=M ** -0.5)
        bias = None
        if case["skew"] > 0:
            p = torch.arange(1, E + 1, dtype=torch.float64) ** -case["skew"]
            bias = torch.log(p / p.sum()).float().to(DEV)
        k = min(case["top_k"], E)
        single = bias is None and ops.forward_int8_single_serves(x, wg, k)
        plan = ops.ForwardInt8Plan(x, wg, k, _capacity(case), logit_bias=bias, single=single)
        return {"case": case, "plan": plan}
    if kind == "bwd":
        T, M, E, dtype = case["tokens"], case["dim"], case["experts"], DTYPES[case["dtype"]]
        cap = _capacity(case)
        routed = ops.route_topk(torch.softmax(_randn(gen, T, E), 1), case["top_k"])
        return {"case": case, "cap": cap, "indices": list(routed["indices"]), "locations": list(routed["locations"]),
                "gates": list(routed["gates"]), "grad": _randn(gen, T, M, dtype=dtype),
                "expert_out": ops.int8_compress(_randn(gen, E * cap, M, dtype=dtype))}
    # a codec: rows of a smooth field (a sinusoid of low frequency and noise), some of them empty slots
    R, M = case["experts"] * case["slots"], case["dim"]
    at = torch.arange(M, device=DEV) * (2 * math.pi / M)
    freq = torch.randint(1, 9, (R, 1), generator=gen, device=DEV)
    phase = torch.rand(R, 1, generator=gen, device=DEV) * (2 * math.pi)
    x = torch.sin(at * freq + phase) + 0.1 * torch.randn(R, M, generator=gen, device=DEV)
    if case["empty"] > 0:
        x *= torch.rand(R, 1, generator=gen, device=DEV) >= case["empty"]
    return {"case": case, "x": x.to(DTYPES[case["dtype"]]).view(case["experts"], case["slots"], M)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "layer":
        layer, x = state["layer"], state["x"]
        if case["mode"] == "infer":
            with torch.no_grad():
                y = layer(x)
            return {"y": y, "l_aux": y.l_aux}
        x.grad = None
        layer.zero_grad(set_to_none=True)
        y = layer(x)
        torch.autograd.backward([y, y.l_aux], [state["grad"], state["loss_weight"].to(y.l_aux.dtype)])
        out = {"grad " + name: p.grad for name, p in layer.named_parameters()}
        out.update({"y": y.detach(), "l_aux": y.l_aux.detach(), "grad x": x.grad})
        return out
    if kind == "route":
        scores, x = state["scores"], state["x"]
        scores.grad = x.grad = None
        crit, l_aux = planmoe_amd.extract_critical(scores, case["top_k"], capacity_factor=case["factor"], alignment=4)
        buffer = planmoe_amd.fast_encode(x, crit)
        y = planmoe_amd.fast_decode(buffer, crit)
        out = {"y": y.detach(), "buffer": buffer.detach(), "l_aux": l_aux.detach(), "indices": crit[1], "locations": crit[2],
               "gates": [g.detach() for g in crit[3]]}
        if case["backward"]:
            y.backward(state["grad"])
            out.update({"grad x": x.grad, "grad scores": scores.grad})
        return out
    if kind == "send":
        return {name: v for name, v in state["plan"].run().items() if v is not None}
    if kind == "bwd":
        indices, locations, E, cap = state["indices"], state["locations"], case["experts"], state["cap"]
        codes, bias, scale, grad_gates = ops.combine_bwd_int8(state["grad"], state["expert_out"], indices, locations, state["gates"], E, cap)
        dx = ops.combine_int8(codes, bias, scale, indices, locations, None, case["tokens"], cap)
        return {"codes": codes, "bias": bias, "scale": scale, "grad gates": grad_gates, "grad x": dx}
    x = state["x"]
    codec = compressor.get_compressor(case["codec"], compressor.get_comm("naive"))
    sent = codec.compress(x)
    codec.adopt(sent)                              # one rank: what arrives is what was sent
    y = codec.decompress(codec.g_output)
    if case["codec"] == "int8":
        return {"codes": sent.view(torch.uint8)[:codec.length], "bias": codec.bias, "scale": codec.scale, "y": y}
    if case["codec"] == "zfp":
        return {"stream": sent.view(torch.uint8)[:codec.length], "y": y}
    return {"flag offsets": codec.flagArrOffsetGlobal, "data offsets": codec.compressedDataOffsetGlobal, "flags": codec.flagArrGlobal,
            "data": codec.compressedDataGlobal, "y": y}


def work(case):
    """Every input read once and every output written once; the products of the tokens, not of the padding."""
    kind = case["kind"]
    s = SIZE[case.get("dtype", "bf16")]
    M, E = case["dim"], case["experts"]
    if kind == "codec":
        n = E * case["slots"] * M
        live = n * (1 - case["empty"])
        coded = {"int8": n, "zfp": n, "lz": live * 4 * 33 / 32}[case["codec"]]
        return {"bytes": 2.0 * (n * s + coded), "flops": 0.0}
    T, k = case["tokens"], min(case["top_k"], case["experts"])
    cap = _capacity(case)
    rows = min(T * k, E * cap)
    plane = T * k * 12
    if kind == "send":
        return {"bytes": float(T * M * 2 + E * M * 2 + E * cap * (M + 4) + plane), "flops": 2.0 * T * M * E}
    if kind == "bwd":
        return {"bytes": float(2 * T * M * s + rows * M + E * cap * (M + 2 * s) + plane + T * k * 4), "flops": 4.0 * rows * M}
    if kind == "route":
        # forward: x in, the buffer out (the caller's), y out; backward: the gradient in, x's gradient out
        n = (2 + (2 if case["backward"] else 0)) * T * M * s + E * cap * M * s + T * E * 4 * (2 if case["backward"] else 1) + 2 * plane
        return {"bytes": float(n), "flops": 2.0 * rows * M * (3 if case["backward"] else 1)}
    H = case["hidden"]
    weights = E * (2 * M * H + H + M) + E * M
    if rows < E:
        weights = weights * rows // E              # experts that no token can reach
    flops = 4.0 * rows * M * H + 2.0 * T * M * E
    if case["mode"] == "infer":
        return {"bytes": float((2 * T * M + weights) * s), "flops": flops}
    return {"bytes": float((4 * T * M + 2 * weights) * s), "flops": 3 * flops}


def tolerance(case):
    kind = case["kind"]
    coarse = case.get("dtype", "bf16") != "fp32"
    if kind == "codec":
        return "exact"                             # codes, streams and what is decoded from them are bits
    if kind == "send":
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-3}      # l_aux and fp32 gates; codes and slots are whole values
    if kind in ("bwd", "route"):
        return {"rel": 1e-2 if coarse else 1e-5, "max": 0.1 if coarse else 1e-3, "differ": 0.0}
    if coarse:
        return {"rel": 1e-2, "max": 0.5}
    # fp32; a lossy codec turns a difference in the last bit into a step of its own now and then
    return {"rel": 1e-3, "max": 0.2} if case["codec"] in ("int8", "zfp") else {"rel": 1e-5, "max": 1e-3}
