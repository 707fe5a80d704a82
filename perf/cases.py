"""The work a user of this package has it do, as cases that can be timed and compared.

Paths, all through the package's public entry points:

* ``layer_decode``   ``gated_deltanet_mixing`` on one new token per sequence: what a generating model calls per layer
* ``layer_prefill``  the same function on a prompt, filling the cache (whole or left-padded batch)
* ``layer_train``    the same function forward and backward: gradients of the projections and of the parameters
* ``decode``         ``fused_recurrent_gated_delta_rule`` on one token per sequence, the state updated in place
* ``forward``        ``chunk_gated_delta_rule``: prompt processing and evaluation, fixed-length or packed sequences
* ``train``          ``chunk_gated_delta_rule`` under autograd: forward and backward of the operator

Head shapes are those of the package's benchmark configurations (K = V = 128; K = 128, V = 256), of the reference's
shipped model configurations (K = 256, V = 512, 2 or 3 heads) and of its smallest tests (K = V = 64); a case with
``HK < H`` shares every head of q and k between H / HK value heads.
"""

from __future__ import annotations

import math

import torch

import lm_engine_amd


BF16, F32 = torch.bfloat16, torch.float32
NORM_EPS = 1e-5
KERNEL_SIZE = 4


def _case(path, B, T, H, K, V, HK=None, N=0, padded=False, dtype="bf16", name=None):
    """``T``: tokens per row (packed: of the one row that holds ``N`` sequences of drawn lengths)."""
    case = dict(path=path, B=B, T=T, H=H, HK=H if HK is None else HK, K=K, V=V, N=N, padded=padded, dtype=dtype)
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # one user's chat, one layer: latency and launches
        _case("layer_decode", 1, 1, 16, 128, 128, name="layer_decode_single"),
        # a serving batch that is not a round number, on one layer of the shipped model
        _case("layer_decode", 53, 1, 2, 256, 512, name="layer_decode_serving"),
        # the decode benchmark: 256 sequences x 32 heads, 512 MiB of state through HBM
        _case("decode", 256, 1, 32, 128, 128, name="decode_256"),
        # a prompt of ordinary length into one layer of the shipped model, length not a multiple of the chunk
        _case("layer_prefill", 1, 777, 2, 256, 512, name="layer_prefill_prompt"),
        # a batch of prompts of different lengths, left-padded, as batched generation starts; heads of q and k shared by two
        # value heads
        _case("layer_prefill", 6, 1500, 16, 128, 128, HK=8, padded=True, name="layer_prefill_padded"),
        # the headline benchmark: a training-sized batch forward
        _case("forward", 4, 4096, 16, 128, 128, name="forward_batch"),
        # packed documents of very different lengths with carried states
        _case("forward", 1, 32768, 16, 128, 128, N=11, name="forward_packed"),
        # one very long context, expanded values
        _case("forward", 1, 65536, 32, 128, 256, name="forward_long"),
        # the exact fp32 path (debugging, small checks): token by token
        _case("forward", 1, 256, 2, 64, 64, dtype="fp32", name="forward_fp32"),
        # training step of the operator at the headline shape
        _case("train", 4, 4096, 16, 128, 128, name="train_batch"),
        # training on packed documents
        _case("train", 1, 32768, 16, 128, 128, N=11, name="train_packed"),
        # training step of one layer of the shipped model at its micro-batch and length
        _case("layer_train", 8, 4096, 2, 256, 512, name="layer_train_shipped"),
    ]  # fmt: skip


_HEADS = ((2, 2, 256, 512), (3, 3, 256, 512), (16, 16, 128, 128), (8, 16, 128, 128), (32, 32, 128, 256), (4, 4, 64, 64))


def _log_uniform(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    path = rng.choice(("layer_decode", "layer_decode", "decode", "layer_prefill", "layer_prefill", "forward", "forward",
                       "forward", "train", "train", "layer_train"))  # fmt: skip
    HK, H, K, V = rng.choice(_HEADS)
    width = H * (K + V)
    if path in ("layer_decode", "decode"):
        most = max(1, min(256, (256 * 32 * 128 * 128) // (H * K * V)))
        return _case(path, _log_uniform(rng, 2 if H == 2 else 1, most), 1, H, K, V, HK=HK)
    if path == "layer_prefill":
        B = rng.choice((1, 1, 2, 3, 5, 8))
        return _case(path, B, _log_uniform(rng, 16, 4096), H, K, V, HK=HK, padded=B > 1 and rng.random() < 0.5)
    if path == "forward" and rng.random() < 0.15:
        return _case(path, rng.choice((1, 2)), _log_uniform(rng, 65, 512), rng.choice((2, 4)), 64, 64, dtype="fp32")
    # tokens of all rows together: at most the largest listed case's work
    tokens = _log_uniform(rng, 130, 32768 if path == "forward" else 20000 * 4096 // max(width, 4096))
    if path != "layer_train" and rng.random() < 0.4:
        return _case(path, 1, tokens, H, K, V, HK=HK, N=rng.randint(2, max(2, min(24, tokens // 100))))
    B = rng.choice((1, 1, 2, 4, 7))
    T = max(65, tokens // B)
    if rng.random() < 0.5:  # training batches are cut to whole chunks more often than not
        T = max(128, T // 64 * 64)
    return _case(path, B, T, H, K, V, HK=HK)


def _lengths(case, seed):
    """Lengths of the packed sequences: uneven, none empty, their sum the row."""
    gen = torch.Generator().manual_seed(seed)
    weights = torch.rand(case["N"], generator=gen) * 0.97 + 0.03
    lengths = (weights / weights.sum() * case["T"]).long().clamp(min=1)
    lengths[lengths.argmax()] += case["T"] - lengths.sum()
    return lengths


def _operator_inputs(case, gen):
    B, T, H, HK, K, V = (case[n] for n in ("B", "T", "H", "HK", "K", "V"))
    dtype = F32 if case["dtype"] == "fp32" else BF16
    normal = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1)  # noqa: E731
    # (rounded to bf16 first, so that the fp32 run of a bf16 case starts from the same values)
    r = lambda x: x.to(BF16).to(dtype)  # noqa: E731
    return dict(
        q=r(unit(normal(B, T, HK, K))), k=r(unit(normal(B, T, HK, K))), v=r(normal(B, T, H, V)),
        g=torch.nn.functional.logsigmoid(3.0 + normal(B, T, H)), beta=r(normal(B, T, H).sigmoid()),
    )  # fmt: skip


def _layer_inputs(case, gen):
    """Outputs of the layer's two projections (the second holds a | b | gate) and its parameters at their initial values."""
    B, T, H, HK, K, V = (case[n] for n in ("B", "T", "H", "HK", "K", "V"))
    dtype = F32 if case["dtype"] == "fp32" else BF16
    normal = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    uniform = lambda *shape: torch.rand(*shape, generator=gen, device="cuda")  # noqa: E731
    r = lambda x: x.to(BF16).to(dtype)  # noqa: E731
    C = 2 * HK * K + H * V
    dt = torch.exp(uniform(H) * (math.log(0.1) - math.log(1e-3)) + math.log(1e-3))
    return dict(
        qkv=r(normal(B, T, C)), ab=r(normal(B, T, 2 * H + H * V)),
        conv_weight=r((uniform(C, 1, KERNEL_SIZE) - 0.5)), conv_bias=r((uniform(C) - 0.5)),
        A_log=torch.log(uniform(H) * 16 + 1e-2), dt_bias=dt + torch.log(-torch.expm1(-dt)), norm_weight=r(1 + 0.1 * normal(V)),
    )  # fmt: skip


def _mix(case, x, cache, attention_mask=None):
    H, HV = case["H"], case["H"] * case["V"]
    a, b, gate = x["ab"].split((H, H, HV), dim=-1)
    return lm_engine_amd.gated_deltanet_mixing(
        x["qkv"], a, b, gate, x["conv_weight"], x["conv_bias"], x["A_log"], x["dt_bias"], x["norm_weight"], NORM_EPS,
        case["HK"], H, case["K"], case["V"], cache=cache, attention_mask=attention_mask)  # fmt: skip


def prepare(case, seed):
    gen = torch.Generator("cuda").manual_seed(seed)
    B, T, H, HK, K, V, path = (case[n] for n in ("B", "T", "H", "HK", "K", "V", "path"))
    dtype = F32 if case["dtype"] == "fp32" else BF16
    state = dict(case=case)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    if path in ("layer_decode", "layer_prefill", "layer_train"):
        state["x"] = x = _layer_inputs(case, gen)
        if path == "layer_decode":  # the cache a prompt has left behind
            C = 2 * HK * K + H * V
            state["cache"] = (normal(B, C, KERNEL_SIZE - 1).to(BF16).to(dtype), 0.02 * normal(B, H, K, V))
        if path == "layer_prefill":
            state["mask"] = None
            if case["padded"]:
                lengths = torch.randint(max(1, T // 3), T + 1, (B,), generator=torch.Generator().manual_seed(seed))
                lengths[0] = T
                state["mask"] = (torch.arange(T)[None, :] >= T - lengths[:, None]).to(torch.int64).cuda()
        if path == "layer_train":
            for leaf in x.values():
                leaf.requires_grad_(True)
            state["d_out"] = normal(B, T, H * V).to(BF16).to(dtype)
        return state
    state["x"] = x = _operator_inputs(case, gen)
    state["cu_seqlens"] = None
    N = B
    if case["N"]:
        N = case["N"]
        state["cu_seqlens"] = torch.nn.functional.pad(_lengths(case, seed).cumsum(0), (1, 0)).to(torch.int32).cuda()
    # decoding, packed documents and long contexts carry a state; a fixed-length batch starts from nothing
    carries = path == "decode" or (path == "forward" and (case["N"] > 0 or T > 8192))
    state["h0"] = 0.02 * normal(N, H, K, V) if carries else None
    if path == "train":
        for leaf in x.values():
            leaf.requires_grad_(True)
        state["d_out"] = normal(B, T, H, V).to(BF16).to(dtype)
    return state


def run(state):
    case, x = state["case"], state["x"]
    path = case["path"]
    if path == "layer_decode":
        with torch.no_grad():
            out, state["cache"] = _mix(case, x, state["cache"])
        return out, state["cache"]
    if path == "layer_prefill":
        with torch.no_grad():
            return _mix(case, x, (None, None), state["mask"])
    if path == "layer_train":
        out, _ = _mix(case, x, None)
        return out.detach(), torch.autograd.grad(out, list(x.values()), state["d_out"])
    if path == "decode":
        with torch.no_grad():
            return lm_engine_amd.fused_recurrent_gated_delta_rule(
                **x, initial_state=state["h0"], output_final_state=True, use_qk_l2norm_in_kernel=True, inplace_state=True)  # fmt: skip
    if path == "forward":
        with torch.no_grad():
            return lm_engine_amd.chunk_gated_delta_rule(
                **x, initial_state=state["h0"], output_final_state=True, cu_seqlens=state["cu_seqlens"])  # fmt: skip
    o, _ = lm_engine_amd.chunk_gated_delta_rule(**x, cu_seqlens=state["cu_seqlens"], use_qk_l2norm_in_kernel=True)
    return o.detach(), torch.autograd.grad(o, list(x.values()), state["d_out"])


def work(case):
    B, T, H, HK, K, V, path = (case[n] for n in ("B", "T", "H", "HK", "K", "V", "path"))
    size = 4 if case["dtype"] == "fp32" else 2
    tokens = B * T
    states = 4 * (case["N"] or B) * H * K * V
    one_token = path in ("layer_decode", "decode") or T <= 64 or size == 4
    # the recurrence token by token, or its chunked form (triangular products at half their dense size)
    flops = tokens * H * (6 * K * V if one_token else 6 * K * V + 64 * (2 * K + 2 * V))
    operands = tokens * (2 * HK * K + H * V)  # q, k, v or the layer's qkv
    gates = tokens * H * (4 + size)  # g, beta
    if path == "decode":
        moved = operands * size + gates + tokens * H * V * size + 2 * states
    elif path == "forward":
        carried = 2 if case["N"] or T > 8192 else 1
        moved = operands * size + gates + tokens * H * V * size + carried * states
    elif path == "train":
        # forward: operands in, o out; backward: operands and d_out in, a gradient for every operand
        moved = 3 * (operands * size + gates) + 2 * tokens * H * V * size
        flops *= 3
    else:
        channels = 2 * HK * K + H * V
        small = channels * (KERNEL_SIZE + 1) * size + H * 8 + V * size
        layer_in = operands * size + tokens * (2 * H + H * V) * size
        layer_out = tokens * H * V * size
        conv_state = B * channels * (KERNEL_SIZE - 1) * size
        if path == "layer_decode":
            moved = layer_in + layer_out + small + 2 * conv_state + 2 * states
        elif path == "layer_prefill":
            moved = layer_in + layer_out + small + conv_state + states
        else:
            moved = 3 * layer_in + 2 * layer_out + 3 * small
            flops *= 3
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """About four times what the bf16 path differs from its own run on the same values in fp32: 3.3e-3 to 4.1e-3 for the
    operator (single elements 0.05 of the larger of value and rms), 4.5e-3 to 5.7e-3 (0.23) for the layer, whose parameter
    gradients cancel over all tokens (2.1e-2 for the two heads' decay)."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["path"] == "layer_train":
        return {"rel": 3e-2, "max": 0.9}
    if case["path"] in ("layer_decode", "layer_prefill"):
        return {"rel": 1.8e-2, "max": 0.65}
    return {"rel": 1.5e-2, "max": 0.2}
