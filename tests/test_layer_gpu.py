"""End to end over the kernels of the layer (convolution -> gates -> operator -> gated norm), chained as
`GatedDeltaNet.forward` chains them (gated_deltanet/module.py:168-242), against the same chain of CPU
oracles; and prefill + decode through the cache against one long prefill."""

import pytest
import torch

import lm_engine_amd
from oracle import recurrent_gated_delta_rule_ref
from oracle.conv_oracle import depthwise_causal_convolution_ref
from oracle.layer_oracle import delta_rule_gates_ref, gated_rmsnorm_ref
from tests.helpers import max_abs, rel_l2


pytestmark = pytest.mark.gpu
BF16, F64 = torch.bfloat16, torch.float64


def _layer_inputs(B, S, HK, HV, DK, DV, seed):
    g = torch.Generator().manual_seed(seed)
    key_dim, value_dim = HK * DK, HV * DV
    qkv = torch.randn(B, S, 2 * key_dim + value_dim, generator=g).to(BF16)
    ab = torch.randn(B, S, 2 * HV + value_dim, generator=g).to(BF16)
    params = dict(
        conv_weight=(0.4 * torch.randn(2 * key_dim + value_dim, 1, 4, generator=g)).to(BF16),
        conv_bias=(0.1 * torch.randn(2 * key_dim + value_dim, generator=g)).to(BF16),
        A_log=torch.log(torch.rand(HV, generator=g) * 4 + 0.1),
        dt_bias=torch.randn(HV, generator=g) - 2.0,
        norm_weight=(1 + 0.1 * torch.randn(DV, generator=g)).to(BF16),
    )
    return qkv, ab, params


def _oracle_chain(qkv, ab, params, HK, HV, DK, DV, cache, neg):
    """The same steps on the CPU in fp64, rounding to bf16 where the kernels hand bf16 tensors on."""
    B, S, _ = qkv.shape
    key_dim, value_dim = HK * DK, HV * DV
    rt = lambda x: x.to(BF16).to(F64)  # noqa: E731
    conv_state, h = cache
    y, conv_state = depthwise_causal_convolution_ref(qkv.to(F64), params["conv_weight"].to(F64), params["conv_bias"].to(F64),
                                                     None if conv_state is None else conv_state.to(F64), None, True)  # fmt: skip
    y = rt(y)
    q, k, v = y.split((key_dim, key_dim, value_dim), dim=-1)
    q = q.reshape(B, S, HK, DK).repeat_interleave(HV // HK, dim=-2)
    k = k.reshape(B, S, HK, DK).repeat_interleave(HV // HK, dim=-2)
    v = v.reshape(B, S, HV, DV)
    a, b, gate = ab[..., :HV], ab[..., HV : 2 * HV], ab[..., 2 * HV :]
    g, beta = delta_rule_gates_ref(a.to(F64), b.to(F64), params["A_log"].to(F64), params["dt_bias"].to(F64), neg)
    g, beta = g.float().to(F64), rt(beta)
    o, h = recurrent_gated_delta_rule_ref(q, k, v, g=g, beta=beta, initial_state=h, output_final_state=True,
                                          use_qk_l2norm_in_kernel=True)  # fmt: skip
    o = rt(o)
    out = gated_rmsnorm_ref(o, gate.to(F64), params["norm_weight"].to(F64), 1e-5)
    return out.flatten(-2), (conv_state, h)


def _gpu_chain(qkv, ab, params, HK, HV, DK, DV, cache, neg, attention_mask=None):
    dev = {n: x.cuda() for n, x in params.items()}
    abd = ab.cuda()
    a, b, gate = abd[..., :HV], abd[..., HV : 2 * HV], abd[..., 2 * HV :]
    return lm_engine_amd.gated_deltanet_mixing(
        qkv.cuda(), a, b, gate, dev["conv_weight"], dev["conv_bias"], dev["A_log"], dev["dt_bias"], dev["norm_weight"],
        1e-5, HK, HV, DK, DV, cache=cache, allow_neg_eigval=neg,
        attention_mask=None if attention_mask is None else attention_mask.cuda())  # fmt: skip


@pytest.mark.parametrize("HK, HV, DK, DV, S", [(2, 4, 128, 128, 200), (4, 4, 64, 64, 130), (2, 2, 128, 256, 70), (4, 8, 128, 128, 40)])
def test_layer_chain_matches_the_chain_of_oracles(HK, HV, DK, DV, S):
    B = 2
    qkv, ab, params = _layer_inputs(B, S, HK, HV, DK, DV, seed=S)
    print(f"case: layer B={B} S={S} heads {HK}/{HV} dims {DK}/{DV}", flush=True)
    ref, (cs_ref, h_ref) = _oracle_chain(qkv, ab, params, HK, HV, DK, DV, (None, None), neg=True)
    out, (cs, h) = _gpu_chain(qkv, ab, params, HK, HV, DK, DV, (None, None), neg=True)
    torch.cuda.synchronize()
    print(f"   out: max-abs {max_abs(out, ref):.3e} rel-L2 {rel_l2(out, ref):.3e}  h: rel-L2 {rel_l2(h, h_ref):.3e}", flush=True)
    assert out.shape == (B, S, HV * DV) and out.dtype == BF16
    # the normalised output is O(1); intermediate bf16 roundings of the two chains differ by an ulp here and there
    assert rel_l2(out, ref) <= 2e-2 and max_abs(out, ref) <= 1e-1
    assert rel_l2(h, h_ref) <= 1e-2
    assert torch.equal(cs.cpu().to(F64), cs_ref)


def test_prefill_then_decode_steps_through_the_cache_match_one_long_prefill():
    B, HK, HV, DK, DV, S, steps = 2, 2, 4, 128, 128, 150, 3
    qkv, ab, params = _layer_inputs(B, S + steps, HK, HV, DK, DV, seed=5)
    full, (cs_full, h_full) = _gpu_chain(qkv, ab, params, HK, HV, DK, DV, (None, None), neg=False)
    out, cache = _gpu_chain(qkv[:, :S], ab[:, :S], params, HK, HV, DK, DV, (None, None), neg=False)
    pieces = [out]
    for i in range(steps):
        out, cache = _gpu_chain(qkv[:, S + i : S + i + 1], ab[:, S + i : S + i + 1], params, HK, HV, DK, DV, cache, neg=False)
        pieces.append(out)
    torch.cuda.synchronize()
    stitched = torch.cat(pieces, dim=1)
    print(f"   stitched vs full: max-abs {max_abs(stitched, full):.3e} rel-L2 {rel_l2(stitched, full):.3e}", flush=True)
    assert rel_l2(stitched, full) <= 1e-2
    assert torch.equal(cache[0], cs_full)
    assert rel_l2(cache[1], h_full) <= 1e-2


def test_no_cache_returns_none():
    qkv, ab, params = _layer_inputs(1, 66, 2, 2, 64, 64, seed=6)
    out, cache = _gpu_chain(qkv, ab, params, 2, 2, 64, 64, None, neg=False)
    assert cache is None and out.shape == (1, 66, 128)


@pytest.mark.parametrize("S", [150, 40])
def test_left_padded_batch_with_attention_mask_equals_unpadded_runs(S):
    # rows padded on the left as the reference batches prompts of different lengths for generation
    B, HK, HV, DK, DV = 3, 2, 4, 128, 128
    lengths = [S, S - 33, 5]
    qkv, ab, params = _layer_inputs(B, S, HK, HV, DK, DV, seed=7)
    mask = torch.zeros(B, S)
    for b, n in enumerate(lengths):
        mask[b, S - n :] = 1
    out, (cs, h) = _gpu_chain(qkv, ab, params, HK, HV, DK, DV, (None, None), neg=False, attention_mask=mask.to(BF16))
    torch.cuda.synchronize()
    for b, n in enumerate(lengths):
        assert torch.all(out[b, : S - n] == 0), f"row {b}: padding must come out as zeros"
        o_b, (cs_b, h_b) = _gpu_chain(qkv[b : b + 1, S - n :], ab[b : b + 1, S - n :], params, HK, HV, DK, DV,
                                      (None, None), neg=False)  # fmt: skip
        print(f"   row {b} len {n}: rel-L2 {rel_l2(out[b : b + 1, S - n :], o_b):.3e}", flush=True)
        # same kernels on the same values; the chunk / recurrent choice may differ between the two calls
        assert rel_l2(out[b : b + 1, S - n :], o_b) <= 1e-2
        assert rel_l2(h[b : b + 1], h_b) <= 1e-2
        assert torch.equal(cs[b : b + 1], cs_b)


def _step_operands(B, HK, HV, DK, DV, dtype, seed):
    qkv, ab, params = _layer_inputs(B, 1, HK, HV, DK, DV, seed=seed)
    g = torch.Generator().manual_seed(seed + 1)
    C = qkv.size(-1)
    cast = lambda x: x.to(dtype).cuda()  # noqa: E731
    cache = (cast(torch.randn(B, C, 3, generator=g)), (0.1 * torch.randn(B, HV, DK, DV, generator=g)).cuda())
    keep = ("A_log", "dt_bias")  # fp32 parameters
    return cast(qkv), cast(ab), {n: (x.cuda() if n in keep else cast(x)) for n, x in params.items()}, cache


def _mix_step(qkv, ab, p, HK, HV, DK, DV, cache, gate=True, neg=True):
    a, b, z = ab[..., :HV], ab[..., HV : 2 * HV], ab[..., 2 * HV :]
    return lm_engine_amd.gated_deltanet_mixing(
        qkv, a, b, z if gate else None, p["conv_weight"], p["conv_bias"], p["A_log"], p["dt_bias"], p["norm_weight"] if gate else None,
        1e-5, HK, HV, DK, DV, cache=cache, allow_neg_eigval=neg)  # fmt: skip


def _watched_host(monkeypatch, step):
    """Puts a recorder in front of the native host path of the layer; ``step`` False: without its one-launch step.  Returns
    the list of what the step answered (None: it left the call to the chain of kernels)."""
    from lm_engine_amd import layer
    from lm_engine_amd._host import host

    answers = []

    class Watched:
        def __getattr__(self, name):
            if name != "layer_step":
                return getattr(host(), name)

            def layer_step(*args):
                answers.append(host().layer_step(*args) if step else None)
                return answers[-1]

            return layer_step

    monkeypatch.setattr(layer, "host", lambda: Watched())
    return answers


# one tile per head (V = 32, 64, 128), tiles of 32, 64 and 128 columns that share a norm through tickets, shared heads of
# q and k, a projection whose gate slice starts off every 16-byte boundary (HV = 1, 2, 3), first token (no state yet)
@pytest.mark.parametrize("dtype", [BF16, torch.float32])
@pytest.mark.parametrize("B, HK, HV, DK, DV", [(1, 4, 4, 64, 32), (3, 2, 4, 128, 64), (5, 1, 3, 256, 128), (2, 2, 2, 128, 96),
                                               (2, 2, 2, 256, 512), (3, 1, 2, 64, 192), (70, 2, 2, 128, 256)])  # fmt: skip
def test_one_launch_step_matches_the_chain_of_kernels(B, HK, HV, DK, DV, dtype, monkeypatch):
    qkv, ab, p, cache = _step_operands(B, HK, HV, DK, DV, dtype, seed=B + DV)
    print(f"case: layer step B={B} heads {HK}/{HV} dims {DK}/{DV} {dtype}", flush=True)

    for gate, start in ((True, cache), (False, cache), (True, (None, None))):
        chained = {}
        for name in ("step", "chain"):
            with monkeypatch.context() as m:
                answers = _watched_host(m, step=name == "step")
                out, c1 = _mix_step(qkv, ab, p, HK, HV, DK, DV, start, gate=gate)
                out2, c2 = _mix_step(qkv, ab, p, HK, HV, DK, DV, c1, gate=gate)  # on the state the first one left
                chained[name] = (out, *c1, out2, *c2)
            assert [x is not None for x in answers] == [name == "step"] * 2, "the kernel under test did not run"
        for name, x, y in zip(("out", "conv", "h", "out2", "conv2", "h2"), chained["step"], chained["chain"]):
            if name.startswith("out"):  # the norm adds its V squares up in another order: at most an ulp of the result
                assert rel_l2(x, y) <= (1e-3 if dtype == BF16 else 1e-6), (name, rel_l2(x, y))
            else:
                assert torch.equal(x, y), name


# every kernel size, parameters in either dtype, with and without a bias; a convolution's state at an odd element gives the bits
# of the same state at an even one
@pytest.mark.parametrize("dtype, w_dtype", [(BF16, BF16), (BF16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("kernel_size, bias, HK, HV, DK, DV", [(2, True, 1, 2, 64, 32), (3, False, 2, 2, 256, 96), (3, True, 1, 2, 128, 256),
                                                               (4, False, 1, 1, 256, 512), (4, True, 1, 1, 64, 128)])  # fmt: skip
def test_one_launch_step_takes_parameters_and_states_as_they_lie(kernel_size, bias, HK, HV, DK, DV, dtype, w_dtype, monkeypatch):
    B = 3
    qkv, ab, p, (conv, h) = _step_operands(B, HK, HV, DK, DV, dtype, seed=kernel_size + DK)
    p["conv_weight"] = p["conv_weight"][..., :kernel_size].contiguous().to(w_dtype)
    p["conv_bias"], p["norm_weight"] = p["conv_bias"].to(w_dtype) if bias else None, p["norm_weight"].to(w_dtype)
    conv = conv[..., : kernel_size - 1].contiguous()
    odd = torch.empty(conv.numel() + 1, dtype=dtype, device="cuda")[1:].view(conv.shape)
    odd.copy_(conv)
    results = []
    for step, state in ((True, conv), (True, odd), (False, conv)):
        with monkeypatch.context() as m:
            answers = _watched_host(m, step=step)
            out, c = _mix_step(qkv, ab, p, HK, HV, DK, DV, (state, h))
        assert [x is not None for x in answers] == [step], "the kernel under test did not run"
        results.append((out, *c))
    for name, x, y, z in zip(("out", "conv", "h"), *results):
        assert torch.equal(x, y), name
        if name == "out":  # (the order of the norm's V squares, as above)
            assert rel_l2(x, z) <= (1e-3 if dtype == BF16 else 1e-6), rel_l2(x, z)
        else:
            assert torch.equal(x, z), name


def test_one_launch_step_under_graph_capture(monkeypatch):
    answers = _watched_host(monkeypatch, step=True)
    HK, HV, DK, DV = 2, 2, 128, 256  # several workgroups per head: tickets in memory of the graph's own
    qkv, ab, p, cache = _step_operands(5, HK, HV, DK, DV, BF16, seed=9)
    with torch.no_grad():
        _mix_step(qkv, ab, p, HK, HV, DK, DV, cache)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out, (conv, h) = _mix_step(qkv, ab, p, HK, HV, DK, DV, cache)
        gen = torch.Generator().manual_seed(3)
        for _ in range(4):
            qkv.copy_(torch.randn(qkv.shape, generator=gen).to(BF16))
            want, (conv_want, h_want) = _mix_step(qkv, ab, p, HK, HV, DK, DV, cache)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want) and torch.equal(conv, conv_want) and torch.equal(h, h_want)
    assert len(answers) == 6 and all(x is not None for x in answers), "the kernel under test did not run"


def test_step_of_rows_whose_norm_overflows_is_that_of_zero_rows(monkeypatch):
    """Finite rows of q and k whose sum of squares is infinite have k^ = q^ = 0: no NaN from k . q."""
    HK, HV, DK, DV = 2, 2, 128, 64
    qkv, ab, p, (_, h) = _step_operands(3, HK, HV, DK, DV, BF16, seed=12)
    p["conv_weight"], p["conv_bias"] = p["conv_weight"].abs(), None
    answers = _watched_host(monkeypatch, step=True)
    outs = []
    for value in (1e25, 0.0):
        x = qkv.clone()
        x[..., : 2 * HK * DK] = value
        out, (_, h_new) = _mix_step(x, ab, p, HK, HV, DK, DV, (None, h))
        outs.append((out, h_new))
    assert len(answers) == 2 and all(x is not None for x in answers)
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1]) and torch.isfinite(outs[0][1]).all()
