"""Parity of the recurrent / decode HIP kernel (through the C ABI) against the CPU oracle."""

import pytest
import torch

import lm_engine_amd
from lm_engine_amd.workloads import get_workload, make_inputs
from oracle import recurrent_gated_delta_rule_ref
from oracle.c_oracle import recurrent_gated_delta_rule_c
from tests.helpers import assert_parity, random_inputs


pytestmark = pytest.mark.gpu


def _to_gpu(inp):
    return {n: (x.cuda() if isinstance(x, torch.Tensor) else x) for n, x in inp.items()}


def _check(inp, dtype, **kwargs):
    print(f"case: recurrent dtype={dtype} shapes q={tuple(inp['q'].shape)} v={tuple(inp['v'].shape)} {kwargs}",
          flush=True)  # fmt: skip
    o_ref, h_ref = recurrent_gated_delta_rule_c(**inp, output_final_state=True, **kwargs)
    o, ht = lm_engine_amd.fused_recurrent_gated_delta_rule(**_to_gpu(inp), output_final_state=True, **kwargs)
    torch.cuda.synchronize()
    assert o.dtype == dtype and ht.dtype == torch.float32
    assert_parity(o.float(), o_ref, dtype, "o")
    assert_parity(ht, h_ref, dtype, "final_state")
    return o, ht


def test_cfg0_ungated_fp32_matches_torch_oracle():
    # configuration 0 of the benchmark contract: B=1, T=256, H=2, K=V=64, fp32, g == 0, zero state
    inp = make_inputs(get_workload(0))
    assert inp["g"] is None and inp["initial_state"] is None
    o_ref, h_ref = recurrent_gated_delta_rule_ref(**inp, output_final_state=True, state_dtype=torch.float64)
    o, ht = lm_engine_amd.fused_recurrent_gated_delta_rule(**_to_gpu(inp), output_final_state=True)
    assert o.shape == (1, 256, 2, 64) and ht.shape == (1, 2, 64, 64)
    assert_parity(o, o_ref, torch.float32, "o")
    assert_parity(ht, h_ref.float(), torch.float32, "final_state")
    # the chunk entry point serves fp32 inputs with the same exact kernel
    o2, h2 = lm_engine_amd.chunk_gated_delta_rule(**_to_gpu(inp), output_final_state=True)
    assert torch.equal(o2, o) and torch.equal(h2, ht)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K, V", [(64, 32), (64, 64), (128, 128), (128, 256), (256, 64), (256, 512)])
def test_head_dims(dtype, K, V):
    inp = random_inputs(B=2, T=9, H=3, K=K, V=V, dtype=dtype, seed=40 + K + V)
    _check(inp, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_l2norm_in_kernel_and_scale(dtype):
    inp = random_inputs(B=2, T=6, H=2, K=128, V=64, dtype=dtype, seed=41, normalize=False, beta_max=2.0)
    _check(inp, dtype, use_qk_l2norm_in_kernel=True, scale=0.3)


def test_ungated_no_beta_no_state():
    inp = random_inputs(B=1, T=12, H=2, K=64, V=64, dtype=torch.bfloat16, seed=42, gated=False, h0=False)
    inp["beta"] = None
    inp["k"] = inp["k"] * 0.5  # beta == 1 with unit keys would make the rule a projection; keep it contractive
    _check(inp, torch.bfloat16)


def test_varlen_packed_sequences():
    lengths = [1, 17, 64, 3, 40]
    inp = random_inputs(B=1, T=sum(lengths), H=2, K=64, V=64, dtype=torch.bfloat16, seed=43, N=len(lengths))
    inp["cu_seqlens"] = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    _check(inp, torch.bfloat16)


def test_varlen_with_empty_sequences():
    lengths = [0, 9, 0, 30, 0]
    inp = random_inputs(B=1, T=sum(lengths), H=2, K=64, V=64, dtype=torch.bfloat16, seed=44, N=len(lengths))
    inp["cu_seqlens"] = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    _check(inp, torch.bfloat16)


def test_left_padded_batch_equals_separate_runs():
    B, T, H = 3, 20, 2
    lengths = [20, 0, 7]
    inp = random_inputs(B=B, T=T, H=H, K=64, V=64, dtype=torch.bfloat16, seed=45)
    gpu = {n: x.cuda() for n, x in inp.items()}
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32).cuda()
    o, ht = lm_engine_amd.fused_recurrent_gated_delta_rule(**gpu, cu_seqlens=cu, output_final_state=True, left_padded=True)
    for b, n in enumerate(lengths):
        assert torch.all(o[b, : T - n] == 0)
        if n == 0:
            assert torch.equal(ht[b], gpu["initial_state"][b])
            continue
        one = {name: x[b : b + 1, T - n :] for name, x in gpu.items() if name != "initial_state"}
        o_b, h_b = lm_engine_amd.fused_recurrent_gated_delta_rule(**one, initial_state=gpu["initial_state"][b : b + 1],
                                                                  output_final_state=True)  # fmt: skip
        assert torch.equal(o[b : b + 1, T - n :], o_b) and torch.equal(ht[b : b + 1], h_b)


def test_strided_views_of_a_fused_projection():
    # q, k, v as the reference layer produces them: slices of one [B, T, 2 H K + H V] projection
    B, T, H, K, V = 2, 5, 2, 64, 128
    gen = torch.Generator().manual_seed(44)
    fused = torch.randn(B, T, 2 * H * K + H * V, generator=gen).to(torch.bfloat16)
    q, k, v = fused.split((H * K, H * K, H * V), dim=-1)
    inp = dict(q=q.view(B, T, H, K), k=k.view(B, T, H, K) * 0.1, v=v.view(B, T, H, V),
               g=-torch.rand(B, T, H, generator=gen), beta=torch.rand(B, T, H, generator=gen).to(torch.bfloat16),
               initial_state=None)  # fmt: skip
    fused_gpu = fused.cuda()
    qg, kg, vg = fused_gpu.split((H * K, H * K, H * V), dim=-1)
    o_ref, h_ref = recurrent_gated_delta_rule_c(**inp, output_final_state=True, use_qk_l2norm_in_kernel=True)
    o, ht = lm_engine_amd.fused_recurrent_gated_delta_rule(
        q=qg.view(B, T, H, K), k=kg.view(B, T, H, K) * 0.1, v=vg.view(B, T, H, V), g=inp["g"].cuda(),
        beta=inp["beta"].cuda(), output_final_state=True, use_qk_l2norm_in_kernel=True)  # fmt: skip
    assert not qg.view(B, T, H, K).is_contiguous()
    assert_parity(o.float(), o_ref, torch.bfloat16, "o")
    assert_parity(ht, h_ref, torch.bfloat16, "final_state")


def test_decode_step_in_place_on_config3_shape():
    # configuration 3: 256 sequences x 32 heads, K = V = 128, fp32 state resident and updated in place
    w = get_workload(3)
    inp = make_inputs(w)
    o_ref, h_ref = recurrent_gated_delta_rule_c(**inp, output_final_state=True)
    gpu = _to_gpu(inp)
    state = gpu["initial_state"]
    ptr = state.data_ptr()
    o, ht = lm_engine_amd.fused_recurrent_gated_delta_rule(**gpu, output_final_state=True, inplace_state=True)
    assert ht.data_ptr() == ptr and o.shape == (256, 1, 32, 128)
    assert_parity(o.float(), o_ref, torch.bfloat16, "o")
    assert_parity(ht, h_ref, torch.bfloat16, "final_state")
    # a second step continues from the updated state
    o_ref2, h_ref2 = recurrent_gated_delta_rule_c(**dict(inp, initial_state=h_ref), output_final_state=True)
    o2, ht2 = lm_engine_amd.fused_recurrent_gated_delta_rule(**gpu, output_final_state=True, inplace_state=True)
    assert_parity(o2.float(), o_ref2, torch.bfloat16, "o (2nd step)")
    assert_parity(ht2, h_ref2, torch.bfloat16, "final_state (2nd step)")


def test_decode_equals_prefill_continuation():
    # prefill T tokens then decode one == run T + 1 tokens at once (same kernel, state carried)
    inp = random_inputs(B=3, T=21, H=2, K=128, V=128, dtype=torch.bfloat16, seed=45)
    gpu = _to_gpu(inp)
    o_all, h_all = lm_engine_amd.fused_recurrent_gated_delta_rule(**gpu, output_final_state=True)
    head = {n: (x[:, :20] if n != "initial_state" else x) for n, x in gpu.items()}
    tail = {n: (x[:, 20:] if n != "initial_state" else x) for n, x in gpu.items()}
    _, h_head = lm_engine_amd.fused_recurrent_gated_delta_rule(**head, output_final_state=True)
    tail["initial_state"] = h_head
    o_tail, h_tail = lm_engine_amd.fused_recurrent_gated_delta_rule(**tail, output_final_state=True)
    assert torch.equal(o_tail, o_all[:, 20:]) and torch.equal(h_tail, h_all)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize(
    "B, H, T, K, V",
    # block edges of the several-token kernel (16 tokens), one to four columns per lane (by the number of workgroups), the
    # few-token walk of the one-token kernel (large batch, T < 12) and its three tile widths
    [(1, 1, 2, 64, 32), (1, 2, 15, 128, 96), (1, 2, 16, 256, 64), (2, 3, 17, 64, 128), (1, 1, 49, 256, 32),
     (40, 16, 13, 64, 64), (70, 16, 12, 128, 128), (66, 16, 3, 64, 64), (33, 8, 11, 128, 256), (20, 16, 2, 256, 512)],
)  # fmt: skip
def test_several_tokens_match_the_oracle_and_the_steps_they_consist_of(dtype, B, H, T, K, V):
    inp = random_inputs(B=B, T=T, H=H, K=K, V=V, dtype=dtype, seed=60 + T, normalize=False)
    o, ht = _check(inp, dtype, use_qk_l2norm_in_kernel=True)
    gpu = _to_gpu(inp)
    cut = T - 1  # the last token on its own: the same bits, whichever kernel and tile width either call runs on
    part = lambda lo, hi: {n: (x[:, lo:hi] if n != "initial_state" else x) for n, x in gpu.items()}  # noqa: E731
    run = lambda x: lm_engine_amd.fused_recurrent_gated_delta_rule(**x, output_final_state=True, use_qk_l2norm_in_kernel=True)  # noqa: E731
    o_head, h_head = run(part(0, cut))
    o_last, h_last = run(dict(part(cut, T), initial_state=h_head))
    assert torch.equal(torch.cat([o_head, o_last], dim=1), o) and torch.equal(h_last, ht)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("l2norm", [False, True])
@pytest.mark.parametrize(
    "lens, H, K, V",
    # V / 4 workgroups per (sequence, head) up to 1024, 512, 256 at K = 64, 128, 256 run as chain, outputs and staging side by
    # side, from 16 tokens on: both sides of these limits, whole and cut blocks, empty and short sequences among longer ones
    [([15], 2, 64, 64), ([16], 2, 64, 64), ([17] * 2, 32, 64, 64), ([17] * 2, 33, 64, 64), ([33], 16, 128, 128),
     ([33], 17, 128, 128), ([48], 2, 256, 512), ([31], 3, 256, 512), ([0, 1, 63, 16, 0, 32, 5], 3, 128, 64)],
)  # fmt: skip
def test_a_few_chains_give_the_bits_of_single_steps(lens, H, K, V, l2norm, dtype):
    N, T = len(lens), sum(lens)
    gpu = _to_gpu(random_inputs(B=1, T=T, H=H, K=K, V=V, dtype=dtype, seed=90 + T, normalize=not l2norm, N=N))
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    h0 = gpu.pop("initial_state")
    state, steps = h0.clone(), h0.clone()
    run = lambda x, h, **kw: lm_engine_amd.fused_recurrent_gated_delta_rule(  # noqa: E731
        **x, initial_state=h, output_final_state=True, use_qk_l2norm_in_kernel=l2norm, **kw)  # fmt: skip
    o, _ = run(gpu, state, cu_seqlens=cu, inplace_state=True)
    for n, begin in enumerate(cu.tolist()[:-1]):
        for t in range(begin, begin + lens[n]):
            want, _ = run({name: x[:, t : t + 1] for name, x in gpu.items()}, steps[n : n + 1], inplace_state=True)
            assert torch.equal(o[:, t : t + 1], want), (n, t)
    assert torch.equal(state, steps)


def test_output_final_state_false_returns_none_and_runs_are_bitwise_repeatable():
    inp = _to_gpu(random_inputs(B=2, T=8, H=2, K=64, V=64, dtype=torch.bfloat16, seed=46))
    o1, none = lm_engine_amd.fused_recurrent_gated_delta_rule(**inp)
    o2, ht = lm_engine_amd.fused_recurrent_gated_delta_rule(**inp, output_final_state=True)
    assert none is None and ht is not None
    assert torch.equal(o1, o2)


def test_inplace_state_is_refused_when_gradients_are_needed():
    inp = _to_gpu(random_inputs(B=1, T=4, H=1, K=64, V=64, dtype=torch.float32, seed=47))
    inp["v"].requires_grad_(True)
    with pytest.raises(ValueError, match="inplace_state"):
        lm_engine_amd.fused_recurrent_gated_delta_rule(**inp, output_final_state=True, inplace_state=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T, magnitude", [(1, 1e25), (1, 3e19), (40, 1e25)])
def test_rows_whose_norm_overflows_count_as_zero_rows(dtype, T, magnitude):
    """x / sqrt(sum x^2 + eps) of a finite row whose sum of squares is infinite is 0 in fp32: such rows of q and k give the
    bits that rows of zeros give, one token or several, and no NaN."""
    inp = _to_gpu(random_inputs(B=2, T=T, H=2, K=128, V=64, dtype=dtype, seed=71, normalize=False))
    huge, zero = dict(inp), dict(inp)
    for n in ("q", "k"):
        huge[n], zero[n] = inp[n].clone(), inp[n].clone()
        huge[n][:, T // 2] = inp[n][:, T // 2].sign() * magnitude
        zero[n][:, T // 2] = 0
    run = lambda x: lm_engine_amd.fused_recurrent_gated_delta_rule(**x, output_final_state=True, use_qk_l2norm_in_kernel=True)  # noqa: E731
    (o, h), (o_zero, h_zero) = run(huge), run(zero)
    assert torch.equal(o, o_zero) and torch.equal(h, h_zero) and torch.isfinite(h).all()


def test_products_of_unnormalised_rows_overflow_only_where_the_result_does():
    """Without l2norm the scale is applied to q before k . q is formed: 2e38 and not infinity times a tenth."""
    z = torch.zeros(1, 1, 1, 64).cuda()
    k, q, v = z + 2e19, z + 2e19, z + 1e-30  # k . q = 64 * 4e38
    o, _ = lm_engine_amd.fused_recurrent_gated_delta_rule(q, k, v, scale=1e-3)
    assert torch.isfinite(o).all() and abs(o.mean().item() / (64 * 4e38 * 1e-3 * 1e-30) - 1) <= 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("lens", [[1] * 70, [1] * 30 + [0, 1, 2, 12, 15, 16, 0, 17, 18, 40] + [3] * 25, [0] * 40 + [64] * 24])
def test_packed_sequences_get_the_bits_of_single_ones_on_either_kernel(lens, inplace, dtype):
    """Decoding (one token each), lengths on both sides of the border between the kernels of one call, empty sequences."""
    H, K, V = 32, 64, 64
    N, T = len(lens), sum(lens)
    gpu = _to_gpu(random_inputs(B=1, T=T, H=H, K=K, V=V, dtype=dtype, seed=83, normalize=False, N=N))
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    h0 = gpu.pop("initial_state")
    own = h0.clone()
    run = lambda x, h, **kw: lm_engine_amd.fused_recurrent_gated_delta_rule(  # noqa: E731
        **x, initial_state=h, output_final_state=True, use_qk_l2norm_in_kernel=True, **kw)
    o, ht = run(gpu, own, cu_seqlens=cu, inplace_state=inplace)
    assert (ht is own) == inplace and (inplace or torch.equal(own, h0))
    begin = 0
    for n, length in enumerate(lens):
        want_h = h0[n : n + 1]
        if length > 0:
            want_o, want_h = run({name: x[:, begin : begin + length] for name, x in gpu.items()}, want_h)
            assert torch.equal(o[:, begin : begin + length], want_o), n
        assert torch.equal(ht[n : n + 1], want_h), n
        begin += length
