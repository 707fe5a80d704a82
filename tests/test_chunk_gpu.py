"""Parity of the chunked-forward HIP kernels (through the C ABI) against the CPU oracle.

Every case feeds the GPU and the oracle the same bf16-rounded tensors; the gate is the one of
the benchmark contract for bf16 inputs: max-abs <= 2e-2 and relative-L2 <= 1e-2 on both the
output and the final state."""

import ctypes
import os

import pytest
import torch

import lm_engine_amd
from lm_engine_amd import _lib, ops
from lm_engine_amd.workloads import get_workload, make_inputs
from oracle.c_oracle import recurrent_gated_delta_rule_c
from tests.dispatch import scan_plan
from tests.helpers import assert_parity, max_abs, random_inputs, rel_l2


pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _to_gpu(inp):
    return {n: (x.cuda() if isinstance(x, torch.Tensor) else x) for n, x in inp.items()}


def _check(inp, label, **kwargs):
    print(f"case: chunk {label} q={tuple(inp['q'].shape)} v={tuple(inp['v'].shape)} {kwargs}", flush=True)
    o_ref, h_ref = recurrent_gated_delta_rule_c(**inp, output_final_state=True, **kwargs)
    o, ht = lm_engine_amd.chunk_gated_delta_rule(**_to_gpu(inp), output_final_state=True, **kwargs)
    torch.cuda.synchronize()
    assert o.dtype == BF16 and ht.dtype == torch.float32
    print(f"   o: max-abs {max_abs(o.float(), o_ref):.3e} rel-L2 {rel_l2(o.float(), o_ref):.3e}   "
          f"ht: max-abs {max_abs(ht, h_ref):.3e} rel-L2 {rel_l2(ht, h_ref):.3e}", flush=True)  # fmt: skip
    assert_parity(o.float(), o_ref, BF16, "o")
    assert_parity(ht, h_ref, BF16, "final_state")
    return o, ht


@pytest.mark.parametrize("T", [65, 128, 130, 321])
def test_sequence_lengths_with_tail_chunks(T):
    _check(random_inputs(B=2, T=T, H=2, K=128, V=128, dtype=BF16, seed=50 + T), f"T={T}")


@pytest.mark.parametrize("K, V", [(64, 32), (64, 64), (128, 64), (128, 256), (256, 128), (256, 512), (128, 160)])
def test_head_dims(K, V):
    _check(random_inputs(B=1, T=200, H=2, K=K, V=V, dtype=BF16, seed=60 + K + V), f"K={K} V={V}")


@pytest.mark.parametrize(
    "B, T, H, K, V, slices_per_workgroup",
    [
        (9, 130, 16, 128, 128, 2),   # 144 chains x 4 slices: more slices than CUs -> two per workgroup
        (20, 130, 16, 128, 128, 4),  # 320 chains x 4 slices -> four per workgroup
        (12, 130, 8, 128, 256, 4),   # 96 chains x 8 slices -> four per workgroup, two groups per chain
        (17, 130, 16, 64, 64, 2),    # 272 chains x 2 slices -> two per workgroup (all of V)
        (30, 130, 16, 128, 96, 1),   # 3 tiles of V: only one slice per workgroup divides them
    ],
)
def test_many_chains_share_records_in_a_workgroup(B, T, H, K, V, slices_per_workgroup):
    # the scan puts 1, 2 or 4 column slices of a chain into one workgroup depending on how many slices
    # there are against the number of CUs (256 on MI355X); ragged length so the last chunk is partial
    inp = random_inputs(B=B, T=T, H=H, K=K, V=V, dtype=BF16, seed=400 + B + V)
    _check(inp, f"B={B} H={H} K={K} V={V}: {slices_per_workgroup} slice(s) per workgroup")


def _sweep_case(i):
    gen = torch.Generator("cpu").manual_seed(9000 + i)
    pick = lambda xs: xs[int(torch.randint(len(xs), (1,), generator=gen))]  # noqa: E731
    K = pick([64, 128])
    V = pick([32, 64, 96, 128, 160, 192, 256])
    H = pick([1, 2, 3, 4, 8])
    T = int(torch.randint(1, 400, (1,), generator=gen))
    B = pick([1, 1, 2, 3, 5])
    return dict(
        B=B, T=T, H=H, K=K, V=V,
        l2norm=pick([False, True]), h0=pick([False, True]), gated=pick([True, True, False]),
        g_mean=pick([-1.0, 1.0, 3.0]), packed=B == 1 and T >= 8 and pick([False, True]),
    )  # fmt: skip


@pytest.mark.parametrize("i", range(int(os.environ.get("GDN_SWEEP_CASES", "16"))))
def test_seeded_sweep_of_shapes_and_options(i):
    # shapes and switches drawn from a seeded generator: head dims, column tiles that do not divide evenly over
    # the workgroup sizes, ragged lengths, packed sequences, state in / no state, ungated, in-kernel l2norm
    c = _sweep_case(i)
    kwargs = dict(use_qk_l2norm_in_kernel=True) if c["l2norm"] else {}
    n_seq, cu = None, None
    if c["packed"]:
        gen = torch.Generator("cpu").manual_seed(9100 + i)
        cuts = sorted(set(int(x) for x in torch.randint(1, c["T"], (3,), generator=gen)))
        cu = torch.tensor([0] + cuts + [c["T"]], dtype=torch.int32)
        n_seq = cu.numel() - 1
    inp = random_inputs(B=c["B"], T=c["T"], H=c["H"], K=c["K"], V=c["V"], dtype=BF16, seed=9200 + i, gated=c["gated"],
                        h0=c["h0"], g_mean=c["g_mean"], normalize=not c["l2norm"], N=n_seq)  # fmt: skip
    if cu is not None:
        inp = dict(inp, cu_seqlens=cu)
    _check(inp, f"sweep {i}: {c}", **kwargs)


def test_short_sequence_single_partial_chunk():
    _check(random_inputs(B=3, T=17, H=2, K=128, V=128, dtype=BF16, seed=70), "T=17")


def test_l2norm_in_kernel_scale_and_negative_eigenvalues():
    # un-normalised q/k with the in-kernel normalisation, beta in (0, 2) as with allow_neg_eigval
    inp = random_inputs(B=2, T=192, H=2, K=128, V=128, dtype=BF16, seed=71, normalize=False, beta_max=2.0)
    _check(inp, "l2norm", use_qk_l2norm_in_kernel=True, scale=0.2)


def test_strong_decay():
    # g around -6 per token: decay factors inside one chunk span e^-380 (underflow to 0 must be harmless)
    _check(random_inputs(B=1, T=256, H=2, K=128, V=128, dtype=BF16, seed=72, g_mean=-6.0), "strong decay")


def test_ungated_no_beta_no_initial_state():
    inp = random_inputs(B=1, T=256, H=2, K=128, V=64, dtype=BF16, seed=73, gated=False, h0=False)
    inp["beta"] = None
    inp["k"] = inp["k"] * 0.5
    _check(inp, "ungated")


def test_fp32_beta_is_accepted():
    inp = random_inputs(B=1, T=130, H=2, K=64, V=64, dtype=BF16, seed=74)
    inp["beta"] = inp["beta"].float()
    _check(inp, "fp32 beta")


def test_varlen_packed_sequences_match_and_equal_separate_runs():
    lengths = [130, 64, 1, 200, 63, 65]
    inp = random_inputs(B=1, T=sum(lengths), H=2, K=128, V=128, dtype=BF16, seed=75, N=len(lengths))
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    o, ht = _check(dict(inp, cu_seqlens=cu), "varlen")
    gpu = _to_gpu(inp)
    for n in range(len(lengths)):
        s, e = int(cu[n]), int(cu[n + 1])
        one = {name: x[:, s:e] for name, x in gpu.items() if name != "initial_state"}
        o_n, h_n = lm_engine_amd.chunk_gated_delta_rule(**one, initial_state=gpu["initial_state"][n : n + 1],
                                                        output_final_state=True)  # fmt: skip
        assert torch.equal(o[:, s:e], o_n), f"sequence {n}: packed and separate outputs differ"
        assert torch.equal(ht[n : n + 1], h_n)


@pytest.mark.parametrize("count, H, V", [(40, 8, 128), (1100, 1, 32)])
def test_varlen_many_sequences_start_longest_first(count, H, V):
    # The scan starts the chains of a packed batch by decreasing length (ranked on the device; batches of more than
    # 1024 sequences keep their order): sequences of equal and of very different lengths, empty ones, more chains
    # than CUs in the first case (two workgroups per CU are accepted for packed batches).
    gen = torch.Generator().manual_seed(count)
    lengths = torch.randint(0, 4, (count,), generator=gen).tolist()
    for i in range(0, count, 7):
        lengths[i] = int(torch.randint(60, 200, (1,), generator=gen))
    lengths[count // 2] = 700
    inp = random_inputs(B=1, T=sum(lengths), H=H, K=64, V=V, dtype=BF16, seed=78, N=count)
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    _check(dict(inp, cu_seqlens=cu), f"varlen, {count} sequences")


@pytest.mark.parametrize("count", [1, 2, 63, 64, 65])
def test_varlen_chunks_are_found_for_any_number_of_sequences(count):
    # the prepare step holds up to 63 prefixes in registers and searches more: empty sequences at the ends and in a row, cut chunks
    gen = torch.Generator().manual_seed(count)
    lengths = torch.randint(0, 200, (count,), generator=gen)
    lengths[torch.rand(count, generator=gen) < 0.3] = 0
    lengths[count // 2] = 129
    inp = random_inputs(B=1, T=int(lengths.sum()), H=2, K=64, V=64, dtype=BF16, seed=79, N=count)
    cu = torch.nn.functional.pad(lengths.cumsum(0), (1, 0)).to(torch.int32)
    _, ht = _check(dict(inp, cu_seqlens=cu), f"varlen, {count} sequences")
    assert torch.equal(ht[lengths == 0].cpu(), inp["initial_state"][lengths == 0])


@pytest.mark.parametrize("lengths, past", [([5], 0), ([64, 0, 64, 130], 0), ([100, 0, 65, 65, 200], 900), ([3] * 60 + [200, 0, 3], 0)])
def test_offsets_of_few_sequences_are_those_of_many(lengths, past):
    # Up to 63 sequences the prepare step forms the offsets and the scan's order, for more a kernel of its own: with empty sequences
    # behind them, the same sequences take the other way.  Equal lengths, empty ones, an end past the batch (cut to it).
    N, extra = len(lengths), 64 - len(lengths)
    inp = _to_gpu(random_inputs(B=1, T=sum(lengths), H=2, K=64, V=64, dtype=BF16, seed=80, N=N))
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    cu[-1] += past
    h0, outcomes = inp.pop("initial_state"), []
    for n in (0, extra):
        leaves = {name: x.clone().requires_grad_(past == 0) for name, x in inp.items() if isinstance(x, torch.Tensor)}
        state = torch.cat([h0, h0[:1].expand(n, -1, -1, -1)]) if n else h0
        o, ht = lm_engine_amd.chunk_gated_delta_rule(**{**inp, **leaves}, initial_state=state, output_final_state=True, cu_seqlens=torch.cat([cu, cu[-1:].expand(n)]).cuda())
        grads = torch.autograd.grad(o.float().square().sum() + ht[:N].sum(), list(leaves.values())) if past == 0 else ()  # (the backward refuses it)
        outcomes.append([o, ht[:N], *grads])
    torch.cuda.synchronize()
    assert all(torch.equal(few, many) for few, many in zip(*outcomes))


@pytest.mark.parametrize("K, V", [(128, 128), (64, 64), (256, 128)])
def test_varlen_with_an_empty_sequence(K, V):
    # a sequence of length 0 has no chunk: its final state is its initial state, and its neighbours are untouched
    lengths = [70, 0, 129, 0]
    inp = random_inputs(B=1, T=sum(lengths), H=2, K=K, V=V, dtype=BF16, seed=77, N=len(lengths))
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    o, ht = _check(dict(inp, cu_seqlens=cu), f"varlen with empty sequences K={K} V={V}")
    assert torch.equal(ht[1].cpu(), inp["initial_state"][1]) and torch.equal(ht[3].cpu(), inp["initial_state"][3])


@pytest.mark.parametrize("K, V", [(128, 128), (256, 128)])
def test_left_padded_batch_equals_separate_runs(K, V):
    # [B, T] batch whose rows are padded on the left; cu_seqlens = prefix sums of the valid lengths
    B, T, H = 4, 200, 2
    lengths = [200, 37, 0, 129]
    inp = random_inputs(B=B, T=T, H=H, K=K, V=V, dtype=BF16, seed=78)
    gpu = _to_gpu(inp)
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32).cuda()
    print(f"case: chunk left-padded lengths {lengths} K={K} V={V}", flush=True)
    o, ht = lm_engine_amd.chunk_gated_delta_rule(**gpu, cu_seqlens=cu, output_final_state=True, left_padded=True)
    for b, n in enumerate(lengths):
        assert torch.all(o[b, : T - n] == 0), f"row {b}: padding must read as zeros"
        if n == 0:
            assert torch.equal(ht[b], gpu["initial_state"][b])
            continue
        one = {name: x[b : b + 1, T - n :] for name, x in gpu.items() if name != "initial_state"}
        o_b, h_b = lm_engine_amd.chunk_gated_delta_rule(**one, initial_state=gpu["initial_state"][b : b + 1], output_final_state=True)
        assert torch.equal(o[b : b + 1, T - n :], o_b), f"row {b}: padded-batch and separate outputs differ"
        assert torch.equal(ht[b : b + 1], h_b)
        # and against the oracle on the valid tokens
        cpu = {name: x[b : b + 1, T - n :] for name, x in inp.items() if name != "initial_state"}
        o_ref, h_ref = recurrent_gated_delta_rule_c(**cpu, initial_state=inp["initial_state"][b : b + 1], output_final_state=True)
        assert_parity(o_b.float(), o_ref, BF16, "o")
        assert_parity(h_b, h_ref, BF16, "final_state")


@pytest.mark.parametrize("B, H, K, V, slices", [(4, 2, 64, 64, 1), (4, 2, 128, 96, 1), (4, 2, 256, 64, 1), (8, 32, 64, 64, 2), (4, 32, 128, 128, 2),
                                                (8, 32, 64, 128, 4), (8, 32, 128, 128, 4), (4, 32, 128, 256, 4)])  # fmt: skip
def test_padding_of_the_output_is_written_on_request_only(B, H, K, V, slices):
    """gdn_chunk_fwd on a left-padded batch, into an output full of NaN: with GDN_FLAG_ZERO_PADDING the padding is zero, without
    it nothing is written there, and the tokens are the same.  Every scan that writes an output: half-slice waves, two and four
    slices per workgroup (one workgroup per chain and several)."""
    cus, chains, tiles = torch.cuda.get_device_properties(0).multi_processor_count, B * H, V // 32
    nw = 1  # as plan_scan counts them
    while K <= 128 and nw < 4 and tiles % (2 * nw) == 0 and chains * (tiles // nw) > cus:
        nw *= 2
    if cus == 256:
        assert nw == slices
    T = 130
    lengths = [T, 0, 1, T - 1, 64, 66, 129, 65][:B]
    gpu = _to_gpu(random_inputs(B=B, T=T, H=H, K=K, V=V, dtype=BF16, seed=79))
    q, k, v, g, beta, h0 = (gpu[n] for n in ("q", "k", "v", "g", "beta", "initial_state"))
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32).cuda()
    dims = ops._check_inputs(q, k, v, g, beta, h0, cu, True)
    lib, stream = _lib.load_library(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print(f"case: padding of the output B={B} H={H} K={K} V={V}", flush=True)
    out = {}
    for flag in (0, _lib.GDN_FLAG_ZERO_PADDING):
        rows = torch.full((B, T, H, V + 8), float("nan"), dtype=BF16, device="cuda")  # (heads with something between them)
        o = rows[..., :V]
        args = ops._fill_args(q, k, v, g, beta, h0, None, o, cu, None, True, False, dims, True)
        args.flags |= flag
        workspace = torch.empty(int(lib.gdn_workspace_bytes(ctypes.byref(args))), dtype=torch.uint8, device="cuda")
        args.workspace, args.workspace_bytes = workspace.data_ptr(), workspace.numel()
        _lib.check_status(lib.gdn_chunk_fwd(ctypes.byref(args), stream), "gdn_chunk_fwd")
        torch.cuda.synchronize()
        assert rows[..., V:].isnan().all()
        out[flag] = o
    for b, n in enumerate(lengths):
        assert out[0][b, : T - n].isnan().all(), f"row {b}: written at the padding"
        assert (out[_lib.GDN_FLAG_ZERO_PADDING][b, : T - n] == 0).all(), f"row {b}: not zero at the padding"
        tokens = [o[b, T - n :] for o in out.values()]
        assert torch.isfinite(tokens[0].float()).all() and torch.equal(*tokens)
    o, _ = lm_engine_amd.chunk_gated_delta_rule(q, k, v, g, beta, initial_state=h0, cu_seqlens=cu, use_qk_l2norm_in_kernel=True, left_padded=True)
    assert torch.equal(o, out[_lib.GDN_FLAG_ZERO_PADDING])


def test_strided_views_of_a_fused_projection():
    B, T, H, K, V = 2, 150, 2, 128, 128
    gen = torch.Generator().manual_seed(76)
    fused = torch.randn(B, T, 2 * H * K + H * V, generator=gen).to(BF16)
    g = -torch.rand(B, T, H, generator=gen) * 0.1
    beta = torch.rand(B, T, H, generator=gen).to(BF16)

    def views(x):
        q, k, v = x.split((H * K, H * K, H * V), dim=-1)
        return q.view(B, T, H, K), k.view(B, T, H, K), v.view(B, T, H, V)

    q, k, v = views(fused)
    o_ref, h_ref = recurrent_gated_delta_rule_c(q=q, k=k, v=v, g=g, beta=beta, output_final_state=True,
                                                use_qk_l2norm_in_kernel=True)  # fmt: skip
    qg, kg, vg = views(fused.cuda())
    assert not qg.is_contiguous()
    o, ht = lm_engine_amd.chunk_gated_delta_rule(q=qg, k=kg, v=vg, g=g.cuda(), beta=beta.cuda(),
                                                 output_final_state=True, use_qk_l2norm_in_kernel=True)  # fmt: skip
    assert_parity(o.float(), o_ref, BF16, "o")
    assert_parity(ht, h_ref, BF16, "final_state")


def test_split_sequence_with_carried_state():
    # prefill [0, 192) then [192, 400) from the carried state == one run over [0, 400)
    inp = _to_gpu(random_inputs(B=2, T=400, H=2, K=128, V=128, dtype=BF16, seed=77))
    o, ht = lm_engine_amd.chunk_gated_delta_rule(**inp, output_final_state=True)
    head = {n: (x[:, :192] if n != "initial_state" else x) for n, x in inp.items()}
    tail = {n: (x[:, 192:] if n != "initial_state" else x) for n, x in inp.items()}
    o1, h1 = lm_engine_amd.chunk_gated_delta_rule(**head, output_final_state=True)
    tail["initial_state"] = h1
    o2, h2 = lm_engine_amd.chunk_gated_delta_rule(**tail, output_final_state=True)
    # 192 is a chunk boundary, so both runs see identical chunks: bitwise equal
    assert torch.equal(torch.cat([o1, o2], dim=1), o) and torch.equal(h2, ht)


def test_chunk_agrees_with_recurrent_kernel_and_is_repeatable():
    inp = _to_gpu(random_inputs(B=2, T=300, H=2, K=128, V=128, dtype=BF16, seed=78))
    o_c, h_c = lm_engine_amd.chunk_gated_delta_rule(**inp, output_final_state=True)
    o_r, h_r = lm_engine_amd.fused_recurrent_gated_delta_rule(**inp, output_final_state=True)
    assert_parity(o_c.float(), o_r.float().cpu(), BF16, "o (chunk vs recurrent kernel)")
    assert_parity(h_c, h_r.cpu(), BF16, "final_state (chunk vs recurrent kernel)")
    o_c2, h_c2 = lm_engine_amd.chunk_gated_delta_rule(**inp, output_final_state=True)
    assert torch.equal(o_c, o_c2) and torch.equal(h_c, h_c2)  # no atomics: bitwise repeatable


def test_output_final_state_false():
    inp = _to_gpu(random_inputs(B=1, T=130, H=2, K=128, V=128, dtype=BF16, seed=79))
    o1, none = lm_engine_amd.chunk_gated_delta_rule(**inp)
    o2, _ = lm_engine_amd.chunk_gated_delta_rule(**inp, output_final_state=True)
    assert none is None and torch.equal(o1, o2)


def test_positional_entry_point_picks_the_kernel_by_length():
    inp = _to_gpu(random_inputs(B=1, T=130, H=2, K=128, V=128, dtype=BF16, seed=80))
    o, ht = lm_engine_amd.gated_delta_rule(inp["q"], inp["k"], inp["v"], inp["beta"], inp["g"], inp["initial_state"])
    o_c, h_c = lm_engine_amd.chunk_gated_delta_rule(**inp, output_final_state=True)
    assert torch.equal(o, o_c) and torch.equal(ht, h_c)
    short = {n: (x[:, :64] if n != "initial_state" else x) for n, x in inp.items()}
    o, ht = lm_engine_amd.gated_delta_rule(short["q"], short["k"], short["v"], short["beta"], short["g"],
                                           short["initial_state"])  # fmt: skip
    o_r, h_r = lm_engine_amd.fused_recurrent_gated_delta_rule(**short, output_final_state=True)
    assert torch.equal(o, o_r) and torch.equal(ht, h_r)


def test_config1_full_size():
    # B=4, T=4096, H=16, K=V=128: the configuration the headline metric is quoted on
    _check(make_inputs(get_workload(1)), "cfg1 full size")


def test_config2_varlen_full_size():
    inp = make_inputs(get_workload(2))
    assert inp["cu_seqlens"][-1].item() == 32768
    _check(inp, f"cfg2 varlen, {inp['cu_seqlens'].numel() - 1} sequences")


def test_config4_long_context_reduced_length():
    # the long-context configuration (H=32, K=128, V=256, h0 random) at T=4096: a quick check of its shape
    _check(make_inputs(get_workload(4, T=4096)), "cfg4 at T=4096")


def test_config4_long_context_full_size():
    # B=1, T=65536, H=32, K=128, V=256, g ~ logsigmoid(N(4, 0.5)): 1024 serial chunks per chain with a long
    # memory, the case where bf16 operand rounding has the most room to accumulate in the state.  Same gate
    # as everywhere (max-abs 2e-2, relative-L2 1e-2 on o and on the final state).
    inp = make_inputs(get_workload(4))
    assert tuple(inp["v"].shape) == (1, 65536, 32, 256)
    o, ht = _check(inp, "cfg4 full size")
    # split at a chunk boundary with the state carried over == one run, bitwise (the kernels are deterministic
    # and a chunk's arithmetic does not depend on its position in the sequence)
    gpu = _to_gpu(inp)
    cut = 64 * 389
    first = {n: (x[:, :cut] if n in ("q", "k", "v", "g", "beta") else x) for n, x in gpu.items()}
    o1, h1 = lm_engine_amd.chunk_gated_delta_rule(**first, output_final_state=True)
    second = {n: (x[:, cut:] if n in ("q", "k", "v", "g", "beta") else x) for n, x in gpu.items()}
    second["initial_state"] = h1
    o2, h2 = lm_engine_amd.chunk_gated_delta_rule(**second, output_final_state=True)
    torch.cuda.synchronize()
    assert torch.equal(torch.cat([o1, o2], dim=1), o), "split run differs from the full run"
    assert torch.equal(h2, ht)


# four slices to a workgroup, whose loaders write the output: one to eight chunks, first and last token of a chunk
@pytest.mark.parametrize("T", [1, 63, 64, 65, 129, 192, 257, 321, 449])
def test_four_slices_at_the_edges_of_chunks(T):
    _check(random_inputs(B=9, T=T, H=16, K=64, V=128, dtype=BF16, seed=120 + T), "four slices")


# two to four chunks, where the compute waves of four slices store the output: with one workgroup to a chain and with two, left-padded rows with
# zeros written at the padding; the loaders' kernel, which longer rows take, gives the same bits for the tokens it shares
@pytest.mark.parametrize("K, B, H, V, T", [(64, 9, 16, 128, 65), (64, 9, 16, 128, 112), (128, 17, 16, 128, 65), (128, 17, 16, 128, 129), (128, 17, 16, 128, 255), (128, 9, 15, 256, 200)])
def test_four_slices_of_few_chunks(K, B, H, V, T):
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert scan_plan(K, B * H, T, V).direct and not scan_plan(K, B * H, T + 256, V).direct
    inp = random_inputs(B=B, T=T + 256, H=H, K=K, V=V, dtype=BF16, seed=140 + T)
    first = {n: (x if n == "initial_state" else x[:, :T].contiguous()) for n, x in inp.items() if isinstance(x, torch.Tensor)}
    o, _ = _check(first, "four slices, few chunks")
    longer, _ = lm_engine_amd.chunk_gated_delta_rule(**_to_gpu(inp))
    whole = T // 64 * 64
    assert torch.equal(longer[:, :whole], o[:, :whole])
    lengths = [T - 29 * b % T for b in range(B)]
    cu = torch.tensor([0, *lengths]).cumsum(0).to(torch.int32).cuda()
    gpu = _to_gpu(first)
    padded, ht = lm_engine_amd.chunk_gated_delta_rule(**gpu, cu_seqlens=cu, output_final_state=True, left_padded=True)
    for b in (0, 1, B - 1):
        assert (padded[b, : T - lengths[b]] == 0).all(), f"row {b}: padding"
        one = {n: (x[b : b + 1].cpu() if n == "initial_state" else x[b : b + 1, T - lengths[b] :].cpu()) for n, x in gpu.items()}
        o_ref, h_ref = recurrent_gated_delta_rule_c(**one, output_final_state=True)
        assert_parity(padded[b : b + 1, T - lengths[b] :].float(), o_ref, BF16, "o")
        assert_parity(ht[b : b + 1], h_ref, BF16, "final_state")


@pytest.mark.parametrize("T", [113, 128])
def test_four_slices_of_two_chunks_through_the_loaders(T):
    _check(random_inputs(B=9, T=T, H=16, K=64, V=128, dtype=BF16, seed=160 + T), "four slices, two chunks")


# K = 256 with up to 256 workgroups of 16 columns: the scan whose keys are split over two waves.  One to seven chunks (its loaders' ring
# fills and drains differently up to five), first and last token of a chunk, one to many column groups, shared heads of q and k
@pytest.mark.parametrize("T, V, HK, H", [(1, 32, 1, 1), (63, 64, 1, 2), (64, 512, 2, 2), (65, 512, 3, 3), (129, 96, 2, 4), (192, 512, 2, 2), (257, 64, 4, 4), (321, 512, 1, 2), (448, 512, 2, 2)])
def test_split_keys_at_the_edges_of_chunks(T, V, HK, H):
    inp = random_inputs(B=2, T=T, H=H, K=256, V=V, dtype=BF16, seed=90 + T)
    q, k = (inp[n][:, :, :HK] for n in ("q", "k"))
    wide = dict(inp, q=q.repeat_interleave(H // HK, dim=2), k=k.repeat_interleave(H // HK, dim=2))
    o_ref, h_ref = recurrent_gated_delta_rule_c(**wide, output_final_state=True)
    gpu = _to_gpu(dict(inp, q=q.contiguous(), k=k.contiguous()))
    print(f"case: split keys T={T} V={V} heads {HK} / {H}", flush=True)
    o, ht = lm_engine_amd.chunk_gated_delta_rule(**gpu, output_final_state=True)
    torch.cuda.synchronize()
    assert_parity(o.float(), o_ref, BF16, "o")
    assert_parity(ht, h_ref, BF16, "final_state")
    if T > 64:  # a chunk's arithmetic does not depend on its place: a run cut behind the first chunk gives the same bits
        part = lambda s: {n: (x[:, s] if n in ("q", "k", "v", "g", "beta") else x) for n, x in gpu.items()}  # noqa: E731
        first, state = lm_engine_amd.chunk_gated_delta_rule(**part(slice(0, 64)), output_final_state=True)
        second, end = lm_engine_amd.chunk_gated_delta_rule(**dict(part(slice(64, None)), initial_state=state), output_final_state=True)
        assert torch.equal(torch.cat([first, second], dim=1), o) and torch.equal(end, ht)


def _half_slices(chains, T, V, packed=False):
    """Past the line of the split keys: half slices, 32 columns to a workgroup."""
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        plan = scan_plan(256, chains, T, V, packed)
        assert plan.half and not plan.split_keys


# the same edges for launches with more workgroups, which keep the half-slice scan: its output, and shared heads of q and k
@pytest.mark.parametrize("T, V, HK, H", [(1, 512, 2, 4), (63, 512, 4, 4), (64, 512, 2, 4), (65, 512, 1, 5), (129, 256, 3, 9), (192, 512, 2, 4), (257, 512, 4, 4), (321, 512, 2, 6), (448, 512, 4, 4)])
def test_half_slices_of_256_keys_at_the_edges_of_chunks(T, V, HK, H):
    _half_slices(4 * H, T, V)
    inp = random_inputs(B=4, T=T, H=H, K=256, V=V, dtype=BF16, seed=170 + T)
    q, k = (inp[n][:, :, :HK].contiguous() for n in ("q", "k"))
    o_ref, h_ref = recurrent_gated_delta_rule_c(**dict(inp, q=q.repeat_interleave(H // HK, dim=2), k=k.repeat_interleave(H // HK, dim=2)), output_final_state=True)
    print(f"case: half slices T={T} V={V} heads {HK} / {H}", flush=True)
    o, ht = lm_engine_amd.chunk_gated_delta_rule(**_to_gpu(dict(inp, q=q, k=k)), output_final_state=True)
    assert_parity(o.float(), o_ref, BF16, "o")
    assert_parity(ht, h_ref, BF16, "final_state")


@pytest.mark.parametrize("lengths", [[70, 0, 129, 0, 64, 65, 1, 200, 33, 128], [3] * 70])
def test_half_slices_of_256_keys_on_packed_sequences(lengths):
    V = 256
    inp = random_inputs(B=1, T=sum(lengths), H=2, K=256, V=V, dtype=BF16, seed=180, N=len(lengths))
    _half_slices(2 * len(lengths), sum(lengths), V, packed=True)
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    _, ht = _check(dict(inp, cu_seqlens=cu), f"half slices, {len(lengths)} sequences")
    empty = torch.tensor(lengths) == 0
    assert torch.equal(ht[empty].cpu(), inp["initial_state"][empty])


def test_half_slices_of_256_keys_on_left_padded_rows():
    B, H, V = 8, 5, 128
    _half_slices(B * H, 130, V)
    test_padding_of_the_output_is_written_on_request_only(B, H, 256, V, 1)
    lengths = [130, 0, 1, 129, 64, 66, 128, 65]
    inp = random_inputs(B=B, T=130, H=H, K=256, V=V, dtype=BF16, seed=181)
    gpu = _to_gpu(inp)
    o, ht = lm_engine_amd.chunk_gated_delta_rule(**gpu, cu_seqlens=torch.tensor([0] + lengths).cumsum(0).to(torch.int32).cuda(), output_final_state=True, left_padded=True)
    for b, n in enumerate(lengths):
        if n == 0:
            assert torch.equal(ht[b].cpu(), inp["initial_state"][b])
            continue
        row = {name: x[b : b + 1] if name == "initial_state" else x[b : b + 1, 130 - n :] for name, x in inp.items()}
        o_ref, h_ref = recurrent_gated_delta_rule_c(**row, output_final_state=True)
        assert_parity(o[b : b + 1, 130 - n :].float(), o_ref, BF16, f"o of row {b}")
        assert_parity(ht[b : b + 1], h_ref, BF16, f"final state of row {b}")


def test_shipped_head_shape_full_size():
    # the head shape of the reference's shipped configurations (k_head_dim 256, v_head_dim 512, 2 heads, micro-batch 8,
    # T = 4096; configs/research/m2rnn/400m-normal/gated-deltanet.yml:60-73): the half-slice scan with a single buffer
    # for the rows of q, 16 chains x 16 slices.  Inputs drawn like configuration 1's.
    inp = make_inputs(get_workload(1, B=8, H=2, K=256, V=512))
    assert tuple(inp["q"].shape) == (8, 4096, 2, 256) and tuple(inp["v"].shape) == (8, 4096, 2, 512)
    o, ht = _check(inp, "K=256, V=512, B=8, T=4096, H=2")
    # split at a chunk boundary with the state carried over == one run, bitwise
    gpu = _to_gpu(inp)
    cut = 64 * 23
    first = {n: (x[:, :cut] if n in ("q", "k", "v", "g", "beta") else x) for n, x in gpu.items()}
    o1, h1 = lm_engine_amd.chunk_gated_delta_rule(**first, output_final_state=True)
    second = {n: (x[:, cut:] if n in ("q", "k", "v", "g", "beta") else x) for n, x in gpu.items()}
    second["initial_state"] = h1
    o2, h2 = lm_engine_amd.chunk_gated_delta_rule(**second, output_final_state=True)
    torch.cuda.synchronize()
    assert torch.equal(torch.cat([o1, o2], dim=1), o), "split run differs from the full run"
    assert torch.equal(h2, ht)
