"""The elementwise steps of the GatedDeltaNet layer on either side of the operator, one HIP kernel each.

* ``delta_rule_gates``  - ``beta = sigmoid(b) [* 2]`` and ``g = -exp(A_log) * softplus(a + dt_bias)``:
  lm_engine/modeling_utils/sequence_mixer_blocks/gated_deltanet/module.py:179-183 with
  ``SoftplusDecayGate.forward(final_exponential=False)``, softplus_decay_gate/module.py:69-96.
* ``gated_rmsnorm``     - ``o_norm(o * silu(gate))``: module.py:238-242 with the RMSNorm of
  lm_engine/modeling_utils/normalization.py:69-124.

Both take the (strided) slices of the layer's projections as they are; there is no torch fallback.
Under autograd the backward of either is one more HIP kernel (``gdn_gated_rmsnorm_bwd``, ``gdn_gates_bwd``).
"""

from __future__ import annotations

import ctypes

import torch

from . import _lib
from ._autograd import kernel_rows, kernel_with_formula_backward
from ._host import host, raw_stream
from .kernels import Kernel, is_kernel_allowed


def _dtype_code(dtype: torch.dtype, what: str) -> int:
    if dtype == torch.bfloat16:
        return _lib.GDN_BF16
    if dtype == torch.float32:
        return _lib.GDN_F32
    raise ValueError(f"{what} must be bfloat16 or float32, got {dtype}")


def _require(x: torch.Tensor, what: str) -> None:
    if not is_kernel_allowed(Kernel.gated_delta_rule):
        raise RuntimeError("Kernel.gated_delta_rule is disabled and this package ships no other implementation")
    if not x.is_cuda:
        raise ValueError(f"{what} must be a device tensor: these kernels run on the GPU only")


def _require_same_device(x: torch.Tensor, what: str, **others) -> None:
    """Ahead of every launch: a tensor elsewhere (on the host, say) would be read through an address that faults the GPU."""
    for name, t in others.items():
        if t is not None and t.device != x.device:
            raise ValueError(f"{name} is on {t.device}, {what} is on {x.device}")


def _token_rows(x: torch.Tensor, width: int, what: str) -> tuple[torch.Tensor, int]:
    """[..., width] view whose leading dims collapse to one token axis with a single stride."""
    if x.size(-1) != width:
        raise ValueError(f"{what}: last dim must be {width}, got {x.size(-1)}")
    if x.stride(-1) != 1:
        x = x.contiguous()
    rows = x.reshape(-1, width) if x.dim() != 2 else x  # a view whenever the leading dims are collapsible
    if rows.stride(-1) != 1:
        rows = rows.contiguous()
    return rows, rows.stride(0) if rows.size(0) > 1 else width


_MASK_BYTES = {torch.int64: 8, torch.int32: 4, torch.uint8: 1, torch.bool: 1}
# The masks that go through one launch.  It is one workgroup of 16 waves, which take a row each and so wait for memory once per 16
# rows; torch's six launches spread them over the chip.  One launch | torch, microseconds on the device (the host asks for 11 | 31),
# int64: 1 x 1024 3.3 | 14, 6 x 1500 4.9 | 15, 64 x 140 6.7 | 14, 17 x 1927 8.6 | 19, 64 x 512 9.4 | 15, 6 x 10922 13 | 20,
# 64 x 1024 14.0 | 15.4; with more rows 96 x 682 17 | 15.5, 128 x 512 16.6 | 14.8, 256 x 35 13.9 | 13.9, 256 x 256 22 | 14, 1024 x 8 49 | 14.
_MASK_ROWS, _MASK_ELEMENTS = 64, 1 << 16


def _one_launch_mask(B: int, S: int, mask_dtype: torch.dtype, dtype: torch.dtype) -> bool:
    return mask_dtype in _MASK_BYTES and dtype in (torch.bfloat16, torch.float32) and 0 < B <= _MASK_ROWS and 0 < B * S <= _MASK_ELEMENTS


def padding_mask(attention_mask: torch.Tensor, dtype: torch.dtype):
    """The integer ``attention_mask`` ``[B, S]`` in ``dtype`` (contiguous) and the prefix sums of its rows' sums, int32 ``[B + 1]``, in
    one launch (``gdn_padding_mask``); the same through torch where that is the faster way or the mask of another type."""
    B, S = attention_mask.shape
    if not attention_mask.is_cuda or not _one_launch_mask(B, S, attention_mask.dtype, dtype):
        seqlens = attention_mask.sum(dim=-1, dtype=torch.int32)  # sequence_packing.py:18-22
        return attention_mask, torch.nn.functional.pad(torch.cumsum(seqlens, dim=0, dtype=torch.int32), (1, 0))
    return _padding_mask_kernel(attention_mask, dtype)


def _padding_mask_kernel(attention_mask, dtype):
    B, S = attention_mask.shape
    mask = torch.empty(B, S, dtype=dtype, device=attention_mask.device)
    prefix = torch.empty(B + 1, dtype=torch.int32, device=attention_mask.device)
    lib = _lib.load_library()
    with torch.cuda.device(attention_mask.device):
        stream = ctypes.c_void_p(torch.cuda.current_stream(attention_mask.device).cuda_stream)
        _lib.check_status(
            lib.gdn_padding_mask(attention_mask.data_ptr(), _MASK_BYTES[attention_mask.dtype], attention_mask.stride(0), attention_mask.stride(1), B, S,
                                 mask.data_ptr(), _dtype_code(dtype, "mask"), prefix.data_ptr(), stream), "gdn_padding_mask")  # fmt: skip
    return mask, prefix


def column_sums(lib, stream, *wanted):
    """``gdn_column_sums``: for every ``(partial [rows, ...] fp32 contiguous, dtype)`` (one or two, the same ``rows``) the sum
    over the first dim in that dtype.  Runs on the caller's current device and stream."""
    if any(dtype not in (torch.bfloat16, torch.float32) for _, dtype in wanted):  # parameters of another type
        return [partial.sum(dim=0).to(dtype) for partial, dtype in wanted]
    args = _lib.GdnColumnSumsArgs()
    results = []
    for j, (partial, dtype) in enumerate(wanted):
        result = torch.empty(partial.shape[1:], dtype=dtype, device=partial.device)
        args.partial[j], args.out[j], args.cols[j] = partial.data_ptr(), result.data_ptr(), result.numel()
        args.out_dtype[j] = _dtype_code(dtype, "gradient")
        results.append(result)
    args.rows, args.arrays = wanted[0][0].size(0), len(wanted)
    _lib.check_status(lib.gdn_column_sums(ctypes.byref(args), stream), "gdn_column_sums")
    return results


def gates_formula(a, b, A_log, dt_bias, allow_neg_eigval):
    """The gates in torch operations: what their backward differentiates."""
    g = -torch.exp(A_log.float()) * torch.nn.functional.softplus(a.float() + dt_bias.float())
    beta = torch.sigmoid(b.float()) * (2.0 if allow_neg_eigval else 1.0)
    return g, beta.to(b.dtype)


def delta_rule_gates(
    a: torch.Tensor, b: torch.Tensor, A_log: torch.Tensor, dt_bias: torch.Tensor, allow_neg_eigval: bool = False
) -> tuple[torch.Tensor, torch.Tensor]:
    """a, b ``[..., H]`` (activation dtype, may be slices of one projection) -> ``(g fp32, beta)`` of the same shape."""

    if torch.compiler.is_compiling():  # a graph is being captured: the kernel goes in as an opaque operator
        from . import _opaque

        return _opaque.delta_rule_gates(a, b, A_log, dt_bias, allow_neg_eigval)

    if a.is_cuda and is_kernel_allowed(Kernel.gated_delta_rule):
        result = host().gates(raw_stream(a.get_device()), a, b, A_log, dt_bias, 2.0 if allow_neg_eigval else 1.0)
        if result is not None:
            return result

    def formula(a, b, A_log, dt_bias):
        return gates_formula(a, b, A_log, dt_bias, allow_neg_eigval)

    kernel = lambda a, b, A_log, dt_bias: _delta_rule_gates(a, b, A_log, dt_bias, allow_neg_eigval)  # noqa: E731
    needs_grad = torch.is_grad_enabled() and any(t.requires_grad for t in (a, b, A_log, dt_bias))
    if needs_grad and a.is_cuda and a.dtype in (torch.bfloat16, torch.float32):
        return _GatesOnKernels.apply(a, b, A_log, dt_bias, allow_neg_eigval)
    return kernel_with_formula_backward(kernel, formula, a, b, A_log, dt_bias)


class _GatesOnKernels(torch.autograd.Function):
    """Forward and backward on the HIP kernels."""

    @staticmethod
    def forward(ctx, a, b, A_log, dt_bias, allow_neg_eigval):
        ctx.save_for_backward(a, b, A_log, dt_bias)
        ctx.allow_neg_eigval = allow_neg_eigval
        result = None
        if is_kernel_allowed(Kernel.gated_delta_rule):
            result = host().gates(raw_stream(a.get_device()), a, b, A_log, dt_bias, 2.0 if allow_neg_eigval else 1.0)
        return _delta_rule_gates(a, b, A_log, dt_bias, allow_neg_eigval) if result is None else result

    @staticmethod
    def backward(ctx, dg, dbeta):
        a, b, A_log, dt_bias = ctx.saved_tensors
        return (*_delta_rule_gates_backward(a, b, A_log, dt_bias, dg, dbeta, ctx.allow_neg_eigval), None)


def _delta_rule_gates_backward(a, b, A_log, dt_bias, dg, dbeta, allow_neg_eigval):
    """``gdn_gates_bwd``: gradients with respect to a, b (contiguous, their dtype), A_log and dt_bias."""
    _require(a, "a")
    if dg is not None and dbeta is not None:
        grads = host().gates_bwd(raw_stream(a.get_device()), a, b, A_log, dt_bias, dg, dbeta, 2.0 if allow_neg_eigval else 1.0)
        if grads is not None:
            return grads
    H = a.size(-1)
    a2, a_stride = _token_rows(a, H, "a")
    b2, b_stride = _token_rows(b, H, "b")
    tokens = a2.size(0)
    dev = a.device
    dg = (torch.zeros(a.shape, dtype=torch.float32, device=dev) if dg is None else dg.to(torch.float32)).contiguous()
    dbeta = (torch.zeros(a.shape, dtype=a.dtype, device=dev) if dbeta is None else dbeta.to(a.dtype)).contiguous()
    da = torch.empty(a.shape, dtype=a.dtype, device=dev)
    db = torch.empty(a.shape, dtype=a.dtype, device=dev)
    if tokens == 0:
        return da, db, torch.zeros_like(A_log), torch.zeros_like(dt_bias)
    blocks = min(1024, max(1, (tokens * H + 255) // 256))
    parts = torch.empty(2, blocks, H, dtype=torch.float32, device=dev)
    A32 = A_log.to(device=dev, dtype=torch.float32).contiguous()
    dt32 = dt_bias.to(device=dev, dtype=torch.float32).contiguous()
    args = _lib.GdnGateBwdArgs()
    args.a, args.b, args.A_log, args.dt_bias = a2.data_ptr(), b2.data_ptr(), A32.data_ptr(), dt32.data_ptr()
    args.dg, args.dbeta, args.da, args.db = dg.data_ptr(), dbeta.data_ptr(), da.data_ptr(), db.data_ptr()
    args.dA_log_partial, args.ddt_bias_partial = parts[0].data_ptr(), parts[1].data_ptr()
    args.a_stride, args.b_stride, args.tokens, args.H = a_stride, b_stride, tokens, H
    args.dtype = _dtype_code(a.dtype, "a, b")
    args.beta_scale = 2.0 if allow_neg_eigval else 1.0
    args.partial_blocks = blocks
    lib = _lib.load_library()
    with torch.cuda.device(dev):
        stream = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
        _lib.check_status(lib.gdn_gates_bwd(ctypes.byref(args), stream), "gdn_gates_bwd")
        # two results that share no storage (an operator's outputs must not alias each other)
        dA_log, ddt_bias = column_sums(lib, stream, (parts[0], A_log.dtype), (parts[1], dt_bias.dtype))
    return da, db, dA_log, ddt_bias


def _delta_rule_gates(a, b, A_log, dt_bias, allow_neg_eigval):
    _require(a, "a")
    H = a.size(-1)
    if b.shape != a.shape or b.dtype != a.dtype:
        raise ValueError("a and b must share shape and dtype")
    if tuple(A_log.shape) != (H,) or tuple(dt_bias.shape) != (H,):
        raise ValueError(f"A_log and dt_bias must be [H] = {(H,)}")
    _require_same_device(a, "a", b=b)
    a2, a_stride = _token_rows(a, H, "a")
    b2, b_stride = _token_rows(b, H, "b")
    A_log = A_log.to(device=a.device, dtype=torch.float32).contiguous()
    dt_bias = dt_bias.to(device=a.device, dtype=torch.float32).contiguous()
    g = torch.empty(a.shape, dtype=torch.float32, device=a.device)
    beta = torch.empty(a.shape, dtype=a.dtype, device=a.device)

    args = _lib.GdnGateArgs()
    args.a, args.b, args.A_log, args.dt_bias = a2.data_ptr(), b2.data_ptr(), A_log.data_ptr(), dt_bias.data_ptr()
    args.g, args.beta = g.data_ptr(), beta.data_ptr()
    args.a_stride, args.b_stride, args.tokens, args.H = a_stride, b_stride, a2.size(0), H
    args.dtype = _dtype_code(a.dtype, "a, b")
    args.beta_scale = 2.0 if allow_neg_eigval else 1.0
    lib = _lib.load_library()
    with torch.cuda.device(a.device):
        stream = ctypes.c_void_p(torch.cuda.current_stream(a.device).cuda_stream)
        _lib.check_status(lib.gdn_gates_fwd(ctypes.byref(args), stream), "gdn_gates_fwd")
    return g, beta


def gated_rmsnorm_formula(o, gate, weight, eps_value):
    """The gated norm in torch operations: what its backward differentiates off the GPU."""
    x = o.float()
    if gate is not None:
        x = x * torch.nn.functional.silu(gate.float().reshape(o.shape))
    y = x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + eps_value)
    if weight is not None:
        y = y * weight.float()
    return (y.to(o.dtype),)


def gated_rmsnorm(
    o: torch.Tensor, gate: torch.Tensor | None, weight: torch.Tensor | None, eps: float | None = None
) -> torch.Tensor:
    """o ``[..., H, V]``; gate the same shape or ``[..., H * V]`` (a slice of a projection) or None;
    weight ``[V]`` or None.  Returns ``rmsnorm(o * silu(gate)) * weight`` over V, shape and dtype of o.
    ``eps=None`` is torch's default for nn.RMSNorm: the machine epsilon of o's dtype."""
    eps_value = float(torch.finfo(o.dtype).eps if eps is None else eps)

    if torch.compiler.is_compiling():  # a graph is being captured: the kernel goes in as an opaque operator
        from . import _opaque

        return _opaque.gated_rmsnorm(o, gate, weight, eps)

    if o.is_cuda and is_kernel_allowed(Kernel.gated_delta_rule):
        result = host().norm(raw_stream(o.get_device()), o, gate, weight, eps_value)
        if result is not None:
            return result

    def formula(o, gate, weight):
        return gated_rmsnorm_formula(o, gate, weight, eps_value)

    kernel = lambda o, gate, weight: (_gated_rmsnorm(o, gate, weight, eps),)  # noqa: E731
    needs_grad = torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (o, gate, weight))
    if needs_grad and o.is_cuda and o.dtype in (torch.bfloat16, torch.float32):
        return _GatedRMSNormOnKernels.apply(o, gate, weight, eps)
    return kernel_with_formula_backward(kernel, formula, o, gate, weight)[0]


class _GatedRMSNormOnKernels(torch.autograd.Function):
    """Forward and backward on the HIP kernels."""

    @staticmethod
    def forward(ctx, o, gate, weight, eps):
        ctx.save_for_backward(o, gate, weight)
        ctx.eps = eps
        y = None
        if is_kernel_allowed(Kernel.gated_delta_rule):
            y = host().norm(raw_stream(o.get_device()), o, gate, weight, float(torch.finfo(o.dtype).eps if eps is None else eps))
        return _gated_rmsnorm(o, gate, weight, eps) if y is None else y

    @staticmethod
    def backward(ctx, dy):
        o, gate, weight = ctx.saved_tensors
        d_o, d_gate, d_weight = _gated_rmsnorm_backward(o, gate, weight, ctx.eps, dy)
        return d_o, d_gate, d_weight, None


def _gated_rmsnorm_backward(o, gate, weight, eps, dy):
    """``gdn_gated_rmsnorm_bwd``: gradients with respect to o, gate (shaped like gate) and weight."""
    _require(o, "o")
    grads = host().norm_bwd(raw_stream(o.get_device()), o, gate, weight, float(torch.finfo(o.dtype).eps if eps is None else eps), dy)
    if grads is not None:
        return grads
    o2, o_stride, g2, g_stride, H, V = _norm_operands(o, gate)
    tokens = o2.size(0)
    dy = kernel_rows(dy.to(o.dtype).contiguous())
    d_o = torch.empty(o.shape, dtype=o.dtype, device=o.device)
    d_gate = None if gate is None else torch.empty(o.shape, dtype=o.dtype, device=o.device)
    blocks = min(2048, max(1, (tokens * H * max(V // 8, 8) + 255) // 256))
    dw_part = torch.empty(blocks, V, dtype=torch.float32, device=o.device)
    w = None if weight is None else weight.contiguous()
    args = _lib.GdnNormBwdArgs()
    args.o, args.dy, args.d_o, args.dweight_partial = o2.data_ptr(), dy.data_ptr(), d_o.data_ptr(), dw_part.data_ptr()
    args.gate = None if g2 is None else g2.data_ptr()
    args.d_gate = None if d_gate is None else d_gate.data_ptr()
    args.weight = None if w is None else w.data_ptr()
    args.o_stride_t, args.gate_stride_t, args.tokens, args.H, args.V = o_stride, g_stride, tokens, H, V
    args.dtype = _dtype_code(o.dtype, "o")
    args.w_dtype = (_lib.GDN_F32 if w is None else _dtype_code(w.dtype, "weight")) | _lib.GDN_NORM_GATE_DWORDS
    args.eps = float(torch.finfo(o.dtype).eps if eps is None else eps)
    args.partial_blocks = blocks
    lib = _lib.load_library()
    with torch.cuda.device(o.device):
        stream = ctypes.c_void_p(torch.cuda.current_stream(o.device).cuda_stream)
        _lib.check_status(lib.gdn_gated_rmsnorm_bwd(ctypes.byref(args), stream), "gdn_gated_rmsnorm_bwd")
        d_weight = None if weight is None else column_sums(lib, stream, (dw_part, weight.dtype))[0]
    return d_o, (None if gate is None else d_gate.reshape(gate.shape)), d_weight


def _norm_operands(o, gate):
    """Token-row views of o and gate for the norm kernels: ``(o2, o_stride, g2, g_stride, H, V)``."""
    _require(o, "o")
    if o.dim() < 2:
        raise ValueError("o must be [..., H, V]")
    H, V = o.shape[-2], o.shape[-1]
    if V % 8 != 0 or V > 512:
        raise ValueError(f"V={V} is not supported (multiple of 8, at most 512)")
    o2, o_stride = _token_rows(o.flatten(-2) if o.is_contiguous() else o.contiguous().flatten(-2), H * V, "o")
    g2, g_stride = None, 0
    if gate is not None:
        if gate.dtype != o.dtype or gate.numel() != o.numel():
            raise ValueError("gate must have the dtype and number of elements of o")
        _require_same_device(o, "o", gate=gate)
        if gate.shape[-2:] == (H, V) and gate.dim() == o.dim():
            gate = gate.flatten(-2) if gate.stride(-2) == V and gate.stride(-1) == 1 else gate.contiguous().flatten(-2)
        g2, g_stride = _token_rows(gate, H * V, "gate")
        if g2.data_ptr() % 4 != 0 or (g_stride * g2.element_size()) % 4 != 0:
            # the kernels read the gate's rows from any 4-byte boundary (a slice behind 2 * H scalars per row has one)
            g2 = g2.contiguous()
            g_stride = H * V
    return o2, o_stride, g2, g_stride, H, V


def _gated_rmsnorm(o, gate, weight, eps):
    o2, o_stride, g2, g_stride, H, V = _norm_operands(o, gate)
    if weight is not None and tuple(weight.shape) != (V,):
        raise ValueError(f"weight must be [V] = {(V,)}")
    _require_same_device(o, "o", weight=weight)
    weight = None if weight is None else weight.contiguous()
    y = torch.empty(o.shape, dtype=o.dtype, device=o.device)

    args = _lib.GdnNormArgs()
    args.o, args.y = o2.data_ptr(), y.data_ptr()
    args.gate = None if g2 is None else g2.data_ptr()
    args.weight = None if weight is None else weight.data_ptr()
    args.o_stride_t, args.gate_stride_t, args.y_stride_t = o_stride, g_stride, H * V
    args.tokens, args.H, args.V = o2.size(0), H, V
    args.dtype = _dtype_code(o.dtype, "o")
    args.w_dtype = (_lib.GDN_F32 if weight is None else _dtype_code(weight.dtype, "weight")) | _lib.GDN_NORM_GATE_DWORDS
    args.eps = float(torch.finfo(o.dtype).eps if eps is None else eps)
    lib = _lib.load_library()
    with torch.cuda.device(o.device):
        stream = ctypes.c_void_p(torch.cuda.current_stream(o.device).cuda_stream)
        _lib.check_status(lib.gdn_gated_rmsnorm_fwd(ctypes.byref(args), stream), "gdn_gated_rmsnorm_fwd")
    return y
