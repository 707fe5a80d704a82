"""``gdn_chunk_bwd_sweeps`` against both sweeps in fp64 (the formulas of lm_engine_amd/backward.py): what the forward and the reverse
sweep save per chunk, and the gradient of the initial state."""

import pytest
import torch

from tests.helpers import rel_l2


C = 64


def _reference(q, k, v, do, g, beta, scale, h0, dht, spans):
    """Per sequence ``(row, start, length)``: S0, V~, dS1, Y of every chunk and dS0, fp64, from the rounded inputs."""
    H, group = v.size(2), v.size(2) // q.size(2)
    out = []
    for n, (row, start, length) in enumerate(spans):
        NC = -(-length // C)
        pad = lambda x: torch.nn.functional.pad(x[row, start : start + length].double().movedim(1, 0), (0, 0, 0, NC * C - length))  # noqa: E731
        qs, ks = (pad(x).repeat_interleave(group, dim=0) for x in (q, k))
        qs, ks = (x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6) for x in (qs, ks))
        qs = qs * scale
        vs, ds = pad(v), pad(do)
        gs, bs = (pad(x[..., None])[..., 0] for x in (g, beta))
        chunks = lambda x: x.reshape(H, NC, C, *x.shape[2:])  # noqa: E731
        qs, ks, vs, ds, gs, bs = (chunks(x) for x in (qs, ks, vs, ds, gs, bs))
        gam = gs.cumsum(-1)
        e, tail, egl = gam.exp(), (gam[..., -1:] - gam).exp(), gam[..., -1].exp()
        E = (gam[..., :, None] - gam[..., None, :]).exp().tril()
        A = (bs[..., None] * E * (ks @ ks.transpose(-1, -2))).tril(-1)
        T = torch.linalg.inv(torch.eye(C, dtype=torch.float64) + A)
        P = E * (qs @ ks.transpose(-1, -2))
        S = h0[n].double() if h0 is not None else torch.zeros(H, q.size(-1), v.size(-1), dtype=torch.float64)
        dS = dht[n].double() if dht is not None else torch.zeros_like(S)
        S0, Vn, dS1, Y = [], [], [None] * NC, [None] * NC
        for c in range(NC):
            S0.append(S)
            Vn.append(T[:, c] @ (bs[:, c, :, None] * (vs[:, c] - e[:, c, :, None] * (ks[:, c] @ S))))
            S = egl[:, c, None, None] * S + (tail[:, c, :, None] * ks[:, c]).transpose(-1, -2) @ Vn[c]
        for c in reversed(range(NC)):
            dS1[c] = dS
            Y[c] = T[:, c].transpose(-1, -2) @ (P[:, c].transpose(-1, -2) @ ds[:, c] + tail[:, c, :, None] * (ks[:, c] @ dS))
            dS = (egl[:, c, None, None] * dS + (e[:, c, :, None] * qs[:, c]).transpose(-1, -2) @ ds[:, c]
                  - (bs[:, c, :, None] * e[:, c, :, None] * ks[:, c]).transpose(-1, -2) @ Y[c])  # fmt: skip
        out.append((S0, Vn, dS1, Y, dS))
    return out


def _rows(sliced, rows, V):  # [.., V / 32, rows, 32] in the memory of [.., rows, V]
    return sliced.reshape(*sliced.shape[:-2], V // 32, rows, 32).transpose(-3, -2).reshape(*sliced.shape[:-2], rows, V).double().cpu()


# one to six chunks (the loaders' ring fills and drains differently up to five), first and last token of a chunk, empty sequences,
# shared heads of q and k, one and several column slices
CASES = [
    *(("rows", [T], K, 64, 2, 2) for K in (64, 128, 256) for T in (1, 63, 64, 65, 128, 192, 257, 384)),
    *(("packed", [100, 0, 64, 1, 333], K, V, 1, 2) for K, V in ((64, 64), (128, 128), (256, 64), (256, 512))),
    *(("padded", [200, 70, 0, 1], K, 128, 3, 3) for K in (64, 128, 256)),
    # enough chains of about one length for workgroups of 64 columns (K = 128)
    *(("rows", [T] * 5, 128, 128, 4, 8) for T in (1, 65, 192, 256, 257, 384, 449)),
    ("rows", [65] * 10, 128, 64, 4, 8),
    ("packed", [100, 0, 64, 1, 333, 300, 257, 320, 130, 384], 128, 192, 4, 8),
    ("padded", [200, 70, 0, 1], 128, 128, 7, 14),
]


@pytest.mark.gpu
@pytest.mark.parametrize("layout, lens, K, V, HK, H", CASES)
def test_sweeps_match_the_formulas(layout, lens, K, V, HK, H):
    from lm_engine_amd import ops

    gen = torch.Generator().manual_seed(sum(lens) + K + V)
    N = len(lens)
    B, T = (1, sum(lens)) if layout == "packed" else (N, max(lens))
    normal = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    q, k, v, do = (normal(B, T, *s).bfloat16() for s in ((HK, K), (HK, K), (H, V), (H, V)))
    g, beta = torch.nn.functional.logsigmoid(3 + normal(B, T, H)), normal(B, T, H).sigmoid().bfloat16()
    h0, dht = 0.1 * normal(N, H, K, V), 0.1 * normal(N, H, K, V)
    starts = [sum(lens[:n]) for n in range(N)]
    spans = [(0, starts[n], lens[n]) if layout == "packed" else (n, T - lens[n], lens[n]) for n in range(N)]
    cu = None if layout == "rows" else torch.tensor([*starts, sum(lens)], dtype=torch.int32).cuda()
    scale, NC = K**-0.5, max(1, -(-max(lens) // C))
    want = _reference(q, k, v, do, g, beta, scale, h0, dht, spans)
    prep, S0, Vn, dS1, Y, dh0 = ops.chunk_bwd_sweeps(*(x.cuda() for x in (q, k, v, do, g, beta)), scale, True, h0.cuda(), cu,
                                                     layout == "padded", dht.cuda(), NC)  # fmt: skip
    S0, dS1 = (_rows(x.view(N, H, NC, K, V), K, V) for x in (S0, dS1))
    Vn, Y = (_rows(x.view(N, H, NC, C, V), C, V) for x in (Vn, Y))
    for n, (s0, vn, ds1, y, ds0) in enumerate(want):
        # operands rounded to bf16 on the way (2^-9 each) and results saved as bf16: the operator's own gate, 1e-2 in the 2-norm
        assert rel_l2(dh0[n].cpu(), ds0) < 1e-2, f"dh0 of sequence {n}"
        for c in range(len(s0)):
            live = min(C, lens[n] - C * c)
            assert rel_l2(S0[n, :, c], s0[c]) < 1e-2, f"state of sequence {n}, chunk {c}"
            assert rel_l2(dS1[n, :, c], ds1[c]) < 1e-2, f"gradient of the state of sequence {n}, chunk {c}"
            assert rel_l2(Vn[n, :, c, :live], vn[c][:, :live]) < 1e-2, f"V~ of sequence {n}, chunk {c}"
            assert rel_l2(Y[n, :, c].flip(-2)[:, :live], y[c][:, :live]) < 1e-2, f"Y of sequence {n}, chunk {c}"
            assert Y[n, :, c].flip(-2)[:, live:].abs().sum() == 0, "rows past the end"  # the chunk-local kernel reads them
        gamma = torch.cat([prep["gamma"].view(N, H, NC * C)[n, :, C * c : C * c + 1] for c in range(len(s0))], dim=1) if s0 else None
        if s0:
            row, start, _ = spans[n]
            first = torch.stack([g[row, start + C * c] for c in range(len(s0))], dim=1)
            assert torch.equal(gamma.cpu(), first), "prefix sums start at the chunk's first token"


@pytest.mark.gpu
def test_output_gradient_with_rows_far_apart():
    # rows of dO further apart than the kernels' 32-bit row arithmetic takes: the same gradients as from a dense dO
    from lm_engine_amd.backward import gated_delta_rule_backward

    T, K, V, apart = 3, 64, 64, (1 << 24) + 64
    gen = torch.Generator().manual_seed(5)
    q, k, v, dense = (torch.randn(1, T, 1, n, generator=gen).to(torch.bfloat16).cuda() for n in (K, K, V, V))
    do = torch.zeros((T - 1) * apart + V, dtype=torch.bfloat16, device="cuda").as_strided((1, T, 1, V), (T * apart, apart, V, 1))
    do.copy_(dense)
    print(f"case: dO rows {apart} apart", flush=True)
    for far, near in zip(*(gated_delta_rule_backward(q, k, v, None, None, d)[:3] for d in (do, dense))):
        assert torch.equal(far, near)


@pytest.mark.gpu
@pytest.mark.parametrize("layout, lens", [("rows", [256, 256]), ("rows", [130]), ("packed", [100, 0, 64, 1, 333]), ("padded", [200, 70, 0, 1])])
@pytest.mark.parametrize("K, V", [(64, 64), (128, 128), (256, 512)])
def test_every_run_of_the_backward_gives_the_same_bits(layout, lens, K, V):
    """Every sum of the sweeps and of the chunk-local kernel has one order.  Enough heads that several workgroups share a CU, ten runs
    (sums through LDS atomics differed in a few entries from one run to the next)."""
    from lm_engine_amd.backward import gated_delta_rule_backward

    gen = torch.Generator().manual_seed(sum(lens) + K)
    N, H = len(lens), 64
    B, T = (1, sum(lens)) if layout == "packed" else (N, max(lens))
    normal = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    q, k, v, do = (normal(B, T, H, n).bfloat16().cuda() for n in (K, K, V, V))
    g, beta = torch.nn.functional.logsigmoid(3 + normal(B, T, H)).cuda(), normal(B, T, H).sigmoid().bfloat16().cuda()
    h0, dht = (0.1 * normal(N, H, K, V).cuda() for _ in range(2))
    cu = None if layout == "rows" else torch.tensor([0, *lens]).cumsum(0).to(torch.int32).cuda()
    print(f"case: ten runs, {layout} {lens} K={K} V={V}", flush=True)
    first = None
    for _ in range(10):
        grads = gated_delta_rule_backward(q, k, v, g, beta, do, dht, initial_state=h0, cu_seqlens=cu, use_qk_l2norm_in_kernel=True,
                                          left_padded=layout == "padded")  # fmt: skip
        first = grads if first is None else first
        for name, a, b in zip(("dq", "dk", "dv", "dg", "dbeta", "dh0"), grads, first):
            assert torch.isfinite(a.float()).all() and torch.equal(a, b), name


@pytest.mark.gpu
@pytest.mark.parametrize("K, V, B, T", [(64, 128, 65, 65), (64, 128, 64, 130), (128, 128, 65, 65), (256, 64, 129, 64)])
def test_sweeps_in_one_launch_give_the_bits_of_smaller_batches(K, V, B, T):
    """One launch or two (K = 64, more workgroups than compute units), side by side or one after the other."""
    from lm_engine_amd import ops

    gen = torch.Generator().manual_seed(B + T)
    q, k, v, do = (torch.randn(B, T, 1, n, generator=gen).bfloat16().cuda() for n in (K, K, V, V))
    g, beta = torch.nn.functional.logsigmoid(3 + torch.randn(B, T, 1, generator=gen)).cuda(), torch.rand(B, T, 1, generator=gen).bfloat16().cuda()
    h0, dht = (0.1 * torch.randn(B, 1, K, V, generator=gen).cuda() for _ in range(2))
    print(f"case: sweeps of {B} x {T} tokens, K={K} V={V}", flush=True)

    def sweeps(rows):
        return ops.chunk_bwd_sweeps(*(x[rows] for x in (q, k, v, do, g, beta)), K**-0.5, True, h0[rows], None, False, dht[rows], (T + 63) // 64)[1:]

    whole, parts = sweeps(slice(0, B)), [sweeps(slice(b, b + 1)) for b in range(B)]
    for i, (name, x) in enumerate(zip(("S0", "V~", "dS1", "Y", "dh0"), whole)):
        assert torch.equal(x, torch.cat([p[i] for p in parts])), name


@pytest.mark.gpu
def test_rows_of_whole_chunks_whatever_the_field_for_tokens_per_row_holds(monkeypatch):
    """Without sequences and without the flag for ragged rows, ``T_rows`` is not read: the layout is that of NC * 64 tokens a row."""
    from lm_engine_amd import _lib, ops

    gen = torch.Generator().manual_seed(6)
    q, k, v, do = (torch.randn(2, 128, 2, 64, generator=gen).bfloat16().cuda() for _ in range(4))
    g, beta = -torch.rand(2, 128, 2, generator=gen).cuda(), torch.rand(2, 128, 2, generator=gen).bfloat16().cuda()
    prep, S0, Vn, dS1, Y, _ = ops.chunk_bwd_sweeps(q, k, v, do, g, beta, 0.125, True, None, None, False, None, 2)
    print("case: chunk-local gradients, T_rows without a meaning", flush=True)

    def gradients(T_rows):
        class Args(_lib.GdnChunkLocalArgs):
            def __init__(self):
                super().__init__()
                self.T_rows = T_rows

        with monkeypatch.context() as m:
            m.setattr(_lib, "GdnChunkLocalArgs", Args)
            return ops.chunk_local_grads(q, k, v, do, prep, Y, Vn, S0, dS1, 0.125, True, sliced=True)

    for T_rows in (65, 100, 127):
        assert all(torch.equal(x, y) for x, y in zip(gradients(T_rows), gradients(0))), T_rows


@pytest.mark.gpu
@pytest.mark.parametrize("layout, lens, bad", [("packed", [100, 64, 0, 1, 133, 70], 1), ("packed", [100, 64, 0, 1, 133, 70], 4), ("padded", [200, 70, 1, 129], 1)])
@pytest.mark.parametrize("K, V", [(64, 64), (128, 128), (256, 512)])
def test_nan_stays_in_its_sequence(layout, lens, bad, K, V):
    """NaN in every token, state and gradient of one sequence, and at the padding: the other sequences' results keep their bits."""
    import lm_engine_amd
    from lm_engine_amd.backward import gated_delta_rule_backward

    gen = torch.Generator().manual_seed(3)
    N, H, padded = len(lens), 3, layout == "padded"
    B, T = (N, max(lens)) if padded else (1, sum(lens))
    normal = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    q, k, v, do = (normal(B, T, H, n).bfloat16().cuda() for n in (K, K, V, V))
    g, beta = torch.nn.functional.logsigmoid(3 + normal(B, T, H)).cuda(), normal(B, T, H).sigmoid().bfloat16().cuda()
    h0, dht = (0.1 * normal(N, H, K, V).cuda() for _ in range(2))
    cu = torch.tensor([0, *lens]).cumsum(0).to(torch.int32).cuda()
    spans = [(n, slice(T - lens[n], T)) if padded else (0, slice(sum(lens[:n]), sum(lens[: n + 1]))) for n in range(N)]
    print(f"case: NaN in sequence {bad} of {layout} {lens} K={K} V={V}", flush=True)

    def results(q, k, v, do, g, beta, h0, dht):
        options = dict(initial_state=h0, cu_seqlens=cu, use_qk_l2norm_in_kernel=True, left_padded=padded)
        o, ht = lm_engine_amd.chunk_gated_delta_rule(q, k, v, g, beta, output_final_state=True, **options)
        dq, dk, dv, dg, dbeta, dh0 = gated_delta_rule_backward(q, k, v, g, beta, do, dht, **options)
        return (o, dq, dk, dv, dg, dbeta), (ht, dh0)

    def poisoned(x):  # everything but the tokens of the good sequences
        y = torch.full_like(x, float("nan"))
        for n, span in enumerate(spans):
            if n != bad:
                y[span] = x[span]
        return y

    states = [x.clone() for x in (h0, dht)]
    for x in states:
        x[bad] = float("nan")
    want, got = results(q, k, v, do, g, beta, h0, dht), results(*map(poisoned, (q, k, v, do, g, beta)), *states)
    for n, span in enumerate(spans):
        if n != bad:
            assert all(torch.equal(a[span], b[span]) and torch.isfinite(a[span].float()).all() for a, b in zip(got[0], want[0]))
            assert all(torch.equal(a[n], b[n]) for a, b in zip(got[1], want[1]))
