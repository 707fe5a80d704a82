"""Everything `GatedDeltaNet.forward` does between its input and output projections, on the HIP kernels.

Follows lm_engine/modeling_utils/sequence_mixer_blocks/gated_deltanet/module.py:168-242 step by step:

    qkv, conv_state = conv1d(qkv, conv_state)            :168-170  -> depthwise_causal_convolution
    q, k, v = split / view                                :172-177  (views; GVA heads are shared inside the operator)
    beta, g = sigmoid(b) [* 2], decay_gate(a)             :179-183  -> delta_rule_gates
    o, h = chunk or fused_recurrent (T <= 64)             :193-222  -> gated_delta_rule kernels
    o = o_norm(o * silu(gate))                            :238-241  -> gated_rmsnorm

For one token per sequence (decoding) all of it is one launch, ``gdn_layer_step``.

With an attention mask the reference packs q, k, v, g, beta into one token stream and unpacks the output
(:185-191, :226-227, sequence_packing.py:25-93; as written there the packed tensors lose the batch
dimension the operator wants and the unpack shape is not the output's).  Here nothing is copied: the mask
becomes the prefix sums of the valid lengths (sequence_packing.py:18-22) and the kernels work on the
left-padded batch in place (``left_padded=True``), writing zeros at the padding as the unpack would.
"""

from __future__ import annotations

import torch

from ._host import host, raw_stream
from .conv import _IN_KERNEL_ACTIVATIONS, depthwise_causal_convolution
from .kernels import Kernel, is_kernel_allowed
from .layer_ops import delta_rule_gates, gated_rmsnorm, padding_mask
from .ops import RECURRENT_MAX_TOKENS, chunk_gated_delta_rule, column_blocks, fused_recurrent_gated_delta_rule, layer_step_workspace


class _SplitChannels(torch.autograd.Function):
    """``qkv.split`` whose backward hands the three gradients on without a copy when they are the column blocks of one tensor
    already (what the operator's backward writes for q, k and v that are); else it concatenates them as split's does."""

    @staticmethod
    def forward(ctx, qkv, num_k_heads, num_v_heads, k_head_dim, v_head_dim):
        B, S, _ = qkv.shape
        ctx.set_materialize_grads(False)
        ctx.shapes = ((B, S, num_k_heads, k_head_dim), (B, S, num_k_heads, k_head_dim), (B, S, num_v_heads, v_head_dim))
        ctx.options = dict(dtype=qkv.dtype, device=qkv.device)
        key_dim = num_k_heads * k_head_dim
        return tuple(x.view(shape) for x, shape in zip(qkv.split((key_dim, key_dim, num_v_heads * v_head_dim), dim=-1), ctx.shapes))

    @staticmethod
    def backward(ctx, *grads):
        if all(d is None for d in grads):
            return None, None, None, None, None
        grads = [torch.zeros(shape, **ctx.options) if d is None else d for d, shape in zip(grads, ctx.shapes)]
        if column_blocks(*grads):
            B, S = grads[0].shape[:2]
            row = sum(d.size(2) * d.size(3) for d in grads)
            joined = grads[0].as_strided((B, S, row), (S * row, row, 1))
        else:
            joined = torch.cat([d.flatten(-2) for d in grads], dim=-1)
        return joined, None, None, None, None


def gated_deltanet_mixing(
    qkv: torch.Tensor,
    a: torch.Tensor,
    b: torch.Tensor,
    gate: torch.Tensor | None,
    conv_weight: torch.Tensor,
    conv_bias: torch.Tensor | None,
    A_log: torch.Tensor,
    dt_bias: torch.Tensor,
    norm_weight: torch.Tensor | None,
    norm_eps: float | None,
    num_k_heads: int,
    num_v_heads: int,
    k_head_dim: int,
    v_head_dim: int,
    cache: tuple[torch.Tensor | None, torch.Tensor | None] | None = None,
    allow_neg_eigval: bool = False,
    scale: float | None = None,
    conv_activation: str | None = "silu",
    attention_mask: torch.Tensor | None = None,
) -> tuple[torch.Tensor, tuple[torch.Tensor, torch.Tensor] | None]:
    """qkv ``[B, S, 2 * num_k_heads * k_head_dim + num_v_heads * v_head_dim]`` (output of qkv_proj),
    a, b ``[B, S, num_v_heads]``, gate ``[B, S, num_v_heads * v_head_dim]`` or None (slices of ab_proj's
    output).  ``cache`` is None (no caching), ``(None, None)`` (start caching) or the pair returned by the
    previous call.  ``attention_mask`` ``[B, S]``: 1 for tokens, 0 for the padding on the left of shorter
    sequences.  Returns ``(o [B, S, num_v_heads * v_head_dim], new cache or None)``."""
    B, S, _ = qkv.shape
    key_dim, value_dim = num_k_heads * k_head_dim, num_v_heads * v_head_dim
    if qkv.size(-1) != 2 * key_dim + value_dim:
        raise ValueError(f"qkv must have {2 * key_dim + value_dim} channels, got {qkv.size(-1)}")
    if num_v_heads % num_k_heads != 0:
        raise ValueError("num_v_heads must be a multiple of num_k_heads")
    use_cache = cache is not None
    conv_state, h = cache if use_cache else (None, None)

    if (S == 1 and use_cache and attention_mask is None and qkv.is_cuda and conv_activation in _IN_KERNEL_ACTIVATIONS
            and is_kernel_allowed(Kernel.gated_delta_rule) and not torch.compiler.is_compiling()):  # fmt: skip
        # decoding: one launch, where the operands are the usual ones (None: they are not, or a gradient is needed)
        device_index = qkv.get_device()
        stream = raw_stream(device_index)
        step = host().layer_step(stream, qkv, a, b, gate, conv_weight, conv_bias, A_log, dt_bias, norm_weight,
                                 torch.finfo(qkv.dtype).eps if norm_eps is None else norm_eps, num_k_heads, num_v_heads, k_head_dim,
                                 v_head_dim, conv_state, h, 2.0 if allow_neg_eigval else 1.0, k_head_dim**-0.5 if scale is None else scale,
                                 _IN_KERNEL_ACTIVATIONS[conv_activation],
                                 lambda pairs, V: layer_step_workspace(device_index, stream, pairs, V))  # fmt: skip
        if step is not None:
            o, conv_state, h = step
            return o, (conv_state, h)

    front = cu_seqlens = None
    if (qkv.is_cuda and conv_activation in _IN_KERNEL_ACTIVATIONS and is_kernel_allowed(Kernel.gated_delta_rule)
            and not torch.compiler.is_compiling()):  # fmt: skip
        # convolution, gates and the mask's prefix sums in one launch, where the operands are the usual ones
        front = host().layer_front(raw_stream(qkv.get_device()), qkv, conv_weight, conv_bias, conv_state, attention_mask, use_cache,
                                   _IN_KERNEL_ACTIVATIONS[conv_activation], a, b, A_log, dt_bias, 2.0 if allow_neg_eigval else 1.0)  # fmt: skip
    if front is not None:
        qkv, conv_state, g, beta, cu_seqlens = front
    else:
        if (attention_mask is not None and attention_mask.dim() == 2 and attention_mask.shape == (B, S) and attention_mask.device == qkv.device
                and is_kernel_allowed(Kernel.gated_delta_rule) and not torch.compiler.is_compiling()):  # fmt: skip
            attention_mask, cu_seqlens = padding_mask(attention_mask, qkv.dtype)
        qkv, conv_state = depthwise_causal_convolution(qkv, conv_weight, conv_bias, conv_state, attention_mask, use_cache,
                                                       conv_activation)  # fmt: skip
    if torch.is_grad_enabled() and qkv.requires_grad and not torch.compiler.is_compiling():
        q, k, v = _SplitChannels.apply(qkv, num_k_heads, num_v_heads, k_head_dim, v_head_dim)
    else:
        q, k, v = qkv.split((key_dim, key_dim, value_dim), dim=-1)
        q = q.view(B, S, num_k_heads, k_head_dim)
        k = k.view(B, S, num_k_heads, k_head_dim)
        v = v.view(B, S, num_v_heads, v_head_dim)
    # grouped value attention (num_v_heads > num_k_heads): the operator reads head h / (num_v_heads / num_k_heads) of q
    # and k for value head h, so the reference's repeat_interleave copies (module.py:175-177) are not made

    if front is None:
        g, beta = delta_rule_gates(a, b, A_log, dt_bias, allow_neg_eigval)

    if attention_mask is not None and cu_seqlens is None:  # (a captured graph; what is no mask of this batch the convolution has refused)
        seqlens = attention_mask.sum(dim=-1, dtype=torch.int32)  # sequence_packing.py:18-22
        cu_seqlens = torch.nn.functional.pad(torch.cumsum(seqlens, dim=0, dtype=torch.int32), (1, 0))

    op = fused_recurrent_gated_delta_rule if S <= RECURRENT_MAX_TOKENS else chunk_gated_delta_rule
    o, h = op(q=q, k=k, v=v, g=g, beta=beta, scale=scale, initial_state=h, output_final_state=use_cache,
              cu_seqlens=cu_seqlens, use_qk_l2norm_in_kernel=True, left_padded=cu_seqlens is not None)  # fmt: skip

    o = gated_rmsnorm(o, gate, norm_weight, norm_eps)
    return o.flatten(-2, -1), ((conv_state, h) if use_cache else None)
