"""Fused expert FFN -- mirror of the reference's experts/ffn.py (two batched GEMMs with bias and
activation between dispatch and combine).  On the GPU in bf16 and fp32 both GEMMs, and the four of their
backward pass, are planmoe_expert_gemm (hand-written kernels for the matrix cores that read either operand
either way round; no library GEMM is called); forward_from_codes() takes the int8 codes of the receive
buffer straight into the first GEMM."""
import torch
from torch.autograd import forward_ad


def _transformed(*tensors):
    """Whether a tensor is under vmap, a functional gradient or forward-mode differentiation: a node of autograd with
    raw pointers behind it cannot follow those."""
    return any(torch._C._functorch.is_functorch_wrapped_tensor(t) or forward_ad.unpack_dual(t).tangent is not None
               for t in tensors)


def row_fits(length, dtype):
    """256 rows of an operand of planmoe_expert_gemm stay under 2 GiB.  (Longer fp32 rows are the library's; bf16 rows
    are refused: the library's batched bf16 products are kept away from transposed operands.)"""
    return dtype != torch.float32 or length * 4 * 256 < 1 << 31


def _kernel_serves(x, w):
    """planmoe_expert_gemm takes bf16 / fp32 operands on the GPU whose row lengths are whole 16-byte pieces."""
    vec = 8 if x.dtype == torch.bfloat16 else 4
    return (x.is_cuda and x.dtype in (torch.bfloat16, torch.float32) and w.dtype == x.dtype and x.dim() == 3 and x.numel() > 0 and
            w.shape[1] % vec == 0 and w.shape[2] % vec == 0 and x.shape[0] == w.shape[0] and x.shape[2] == w.shape[1] and
            row_fits(max(w.shape[1:]), x.dtype) and not torch.is_autocast_enabled(x.device.type))


def aligned(t):
    """t as the kernels read it: contiguous, 16-byte aligned.  (A view of a flat buffer of parameters or rows begins
    anywhere; it is copied for the product.)"""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


class _BatchedLinear(torch.autograd.Function):
    """y = act(x @ w + bias) over experts: x [E, R, in], w [E, in, out] (as the reference stores it),
    bias [E, out], act = relu or nothing; torch.add(torch.matmul(x, w), bias.unsqueeze(1)) of
    experts/ffn.py:77-79 with its roundings.  All three products read their operands as they lie in
    memory.  dbias sums in fp32."""

    @staticmethod
    def forward(ctx, x, w, bias, relu):
        from . import ops
        x, w = x.contiguous(), w.contiguous()
        y = ops.expert_gemm('nn', aligned(x), aligned(w), None if bias is None else bias.contiguous(), relu=relu)
        ctx.save_for_backward(x, w, y if relu else None)
        ctx.relu, ctx.has_bias = relu, bias is not None
        return y

    @staticmethod
    def backward(ctx, gy):
        from . import ops
        x, w, y = ctx.saved_tensors
        if torch.is_grad_enabled() and gy.dtype == torch.float32:
            # a gradient that is differentiated in turn: the same products where autograd sees them.  (Not in 16 bits: the
            # library's batched products of that kind are kept away from transposed operands)
            if ctx.relu:
                gy = gy * (y > 0)
            return (torch.matmul(gy, w.transpose(1, 2)) if ctx.needs_input_grad[0] else None,
                    torch.matmul(x.transpose(1, 2), gy) if ctx.needs_input_grad[1] else None,
                    gy.sum(dim=1) if ctx.has_bias and ctx.needs_input_grad[2] else None, None)
        if ctx.relu:
            gy = torch.ops.aten.threshold_backward(gy.contiguous(), y, 0.0)      # relu's own backward: one pass over dy and y
        gy = aligned(gy)
        dx = dw = db = None
        if ctx.needs_input_grad[0]:
            dx = ops.expert_gemm('nt', gy, aligned(w))              # [E, R, out] x [E, in, out]^T
        if ctx.needs_input_grad[1]:
            dw = ops.expert_gemm('tn', aligned(x), gy)              # x^T dy
        if ctx.has_bias and ctx.needs_input_grad[2]:
            db = gy.sum(dim=1, dtype=torch.float32).to(gy.dtype)
        return dx, dw, db, None


class FusedExpertsNetwork(torch.nn.Module):
    # experts/ffn.py:13-82, one GPU (no expert sharding)
    def __init__(self, hidden_size_per_expert, activation_fn=None, activation_fn_with_self=None,
                 output_dim=None):
        super().__init__()
        self.hidden_size_per_expert = hidden_size_per_expert
        self.output_dim = output_dim
        if activation_fn_with_self is not None:
            assert activation_fn is None, "Option `activation_fn_with_self` has been specified, please keep exactly one of them."
            activation_fn = lambda x: activation_fn_with_self(x, self)
        self._relu = activation_fn is None          # the default activation: the first GEMM applies it itself
        if activation_fn is None:
            activation_fn = lambda x: torch.nn.functional.relu(x)
        self.activation_fn = activation_fn

    def update(self, ctx):
        model_dim = ctx.model_dim
        local_experts = ctx.num_local_experts
        hidden = self.hidden_size_per_expert
        out = self.output_dim or model_dim
        # parameter names and shapes as the reference's (ffn.py:33-56): fc1 [E, model_dim, hidden],
        # fc2 [E, hidden, out], so that its state dicts load here
        fc1_w = torch.empty(local_experts, model_dim, hidden)
        fc2_w = torch.empty(local_experts, hidden, out)
        fc1_b = torch.empty(local_experts, hidden)
        fc2_b = torch.empty(local_experts, out)
        for i in range(local_experts):
            fc1 = torch.nn.Linear(model_dim, hidden)
            fc2 = torch.nn.Linear(hidden, out)
            fc1_w[i], fc1_b[i] = fc1.weight.t(), fc1.bias
            fc2_w[i], fc2_b[i] = fc2.weight.t(), fc2.bias
        self.batched_fc1_w = torch.nn.Parameter(fc1_w)
        self.batched_fc2_w = torch.nn.Parameter(fc2_w)
        self.batched_fc1_bias = torch.nn.Parameter(fc1_b)
        self.batched_fc2_bias = torch.nn.Parameter(fc2_b)
        self._fc1_k_major = None

    # a batched library GEMM (the dtypes and sizes the kernels do not serve) is not issued above this many
    # multiply-adds: torch's batched kernels with a transposed view as the right operand (what the backward
    # pass of a batched product makes) have faulted the GPU; large products go one expert at a time
    LIBRARY_BATCHED_LIMIT = 1 << 32

    def _linear(self, x, w, bias, relu):
        if _kernel_serves(x, w) and not (x.dtype == torch.float32 and _transformed(x, w, bias)):
            return _BatchedLinear.apply(x, w, bias, relu)
        if x.is_cuda and x.shape[0] > 1 and x.shape[0] * x.shape[1] * w.shape[1] * w.shape[2] > self.LIBRARY_BATCHED_LIMIT:
            y = torch.stack([torch.addmm(bias[e], x[e], w[e]) for e in range(x.shape[0])])
        else:
            y = torch.add(torch.matmul(x, w), bias.unsqueeze(1))
        return torch.nn.functional.relu(y) if relu else y

    def forward(self, x, ctx):
        # experts/ffn.py:63-82
        y = self._linear(x, self.batched_fc1_w, self.batched_fc1_bias, self._relu)
        if not self._relu:
            y = self.activation_fn(y)
        return self._linear(y, self.batched_fc2_w, self.batched_fc2_bias, False)

    _own_forward, _own_linear = forward, _linear        # (as defined here: overlap.native_call asks whether they still are)

    def forward_from_codes(self, codes, bias, scale, exact=True):
        """The same forward with the int8 codes of the receive buffer as input (inference: no autograd
        through the first GEMM): the GEMM reads the codes, so the decompressed [E, C, model_dim]
        tensor is never written.  exact=True (the default): planmoe_ffn_fc1_int8 multiplies the
        decompressor's very values, so the result is that of decompress + GEMM up to the GEMM's
        summation order.  exact=False: planmoe_ffn_fc1_int8_affine puts the codes themselves on the
        matrix cores and applies scale / bias in the epilogue; it skips the decompressor's three
        roundings per element, which is about an ulp of the result for rows whose range is
        comparable to their offset and more than that where |bias| >> scale or the weights'
        column sum cancels -- an approximation to opt into, 1.4 x faster.
        bf16; model_dim % 64 == 0, hidden % 128 == 0."""
        from . import ops
        w = self.batched_fc1_w
        cached = self._fc1_k_major
        key = (w._version, w.data_ptr(), w.device, w.dtype)     # (.data swaps change the pointer, not the version)
        if cached is None or cached[0] != key:
            wk = w.detach().transpose(1, 2).contiguous()                        # [E, hidden, model_dim]
            cached = (key, wk, None if exact else ops.ffn_weight_colsum(wk))
            self._fc1_k_major = cached
        if not exact and cached[2] is None:
            cached = (key, cached[1], ops.ffn_weight_colsum(cached[1]))
            self._fc1_k_major = cached
        if exact:
            y = ops.ffn_fc1_int8(codes, bias, scale, cached[1], self.batched_fc1_bias.detach())
        else:
            y = ops.ffn_fc1_int8_affine(codes, bias, scale, cached[1], cached[2], self.batched_fc1_bias.detach())
        y = self.activation_fn(y)
        return self._linear(y, self.batched_fc2_w, self.batched_fc2_bias, False)


ExpertModule = FusedExpertsNetwork
