"""Parity of the gates and gated-RMSNorm kernels (through the C ABI) against the CPU oracle.
Gates: fp32 outputs within 1e-5 relative; bf16 outputs within max-abs 2e-2 and relative-L2 1e-2."""

import pytest
import torch

import lm_engine_amd
from oracle.layer_oracle import delta_rule_gates_ref, gated_rmsnorm_ref
from tests.helpers import max_abs, rel_l2


pytestmark = pytest.mark.gpu
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("neg", [False, True])
def test_gates_on_slices_of_one_projection(dtype, neg):
    B, T, H, V = 2, 77, 6, 16
    g = torch.Generator().manual_seed(3)
    ab = (3 * torch.randn(B, T, 2 * H + H * V, generator=g)).to(dtype)  # the layer's ab_proj output: a | b | gate
    ab[0, 0, 0] = 40.0  # softplus threshold branch
    a, b = ab[..., :H], ab[..., H : 2 * H]
    A_log = torch.log(torch.rand(H, generator=g) * 16 + 1e-3)
    dt_bias = torch.randn(H, generator=g)
    print(f"case: gates {dtype} neg={neg} a stride {a.stride()}", flush=True)
    g_ref, beta_ref = delta_rule_gates_ref(a.to(F64), b.to(F64), A_log.to(F64), dt_bias.to(F64), neg)
    abd = ab.cuda()
    g_out, beta = lm_engine_amd.delta_rule_gates(abd[..., :H], abd[..., H : 2 * H], A_log.cuda(), dt_bias.cuda(), neg)
    torch.cuda.synchronize()
    assert g_out.dtype == F32 and beta.dtype == dtype and g_out.shape == a.shape and beta.shape == a.shape
    assert (g_out <= 0).all()
    torch.testing.assert_close(g_out.cpu().to(F64), g_ref, rtol=1e-5, atol=1e-6)
    if dtype == F32:
        torch.testing.assert_close(beta.cpu().to(F64), beta_ref, rtol=1e-5, atol=1e-6)
    else:
        assert max_abs(beta, beta_ref) <= 2e-2 and rel_l2(beta, beta_ref) <= 1e-2


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("V", [64, 96, 128, 256, 512])
@pytest.mark.parametrize("gated", [False, True])
def test_gated_rmsnorm(dtype, V, gated):
    B, T, H = 2, 45, 3
    g = torch.Generator().manual_seed(V)
    o = torch.randn(B, T, H, V, generator=g).to(dtype)
    proj = torch.randn(B, T, 8 + H * V, generator=g).to(dtype)  # gate is a slice of a wider projection
    gate = proj[..., 8:] if gated else None
    w = (1 + 0.1 * torch.randn(V, generator=g)).to(dtype)
    print(f"case: gated_rmsnorm {dtype} V={V} gated={gated}", flush=True)
    y_ref = gated_rmsnorm_ref(o.to(F64), None if gate is None else gate.to(F64), w.to(F64), 1e-5)
    pd = proj.cuda()
    y = lm_engine_amd.gated_rmsnorm(o.cuda(), pd[..., 8:] if gated else None, w.cuda(), 1e-5)
    torch.cuda.synchronize()
    assert y.dtype == dtype and y.shape == o.shape
    if dtype == F32:
        torch.testing.assert_close(y.cpu().to(F64), y_ref, rtol=1e-5, atol=1e-5)
    else:
        assert max_abs(y, y_ref) <= 2e-2 * max(1.0, float(y_ref.abs().max())) and rel_l2(y, y_ref) <= 1e-2
    # the [.., H, V] view of the gate slice is accepted as well
    if gated:
        y2 = lm_engine_amd.gated_rmsnorm(o.cuda(), pd[..., 8:].view(B, T, H, V), w.cuda(), 1e-5)
        assert torch.equal(y, y2)


def test_gate_slice_off_a_16_byte_boundary():
    # with 2 or 3 heads the gate columns start 2 * H elements into the projection: 8 or 12 bytes in bf16
    B, T, H, V = 2, 33, 3, 512
    g = torch.Generator().manual_seed(9)
    o = torch.randn(B, T, H, V, generator=g).to(BF16)
    proj = torch.randn(B, T, 2 * H + H * V, generator=g).to(BF16)
    y_ref = gated_rmsnorm_ref(o.to(F64), proj[..., 2 * H :].to(F64), None, 1e-6)
    y = lm_engine_amd.gated_rmsnorm(o.cuda(), proj.cuda()[..., 2 * H :], None, 1e-6)
    assert rel_l2(y, y_ref) <= 1e-2


@pytest.mark.parametrize("dtype,offset", [(BF16, 2), (BF16, 4), (BF16, 6), (BF16, 7), (F32, 1), (F32, 2), (F32, 3)])
@pytest.mark.parametrize("V", [64, 504])
def test_gate_rows_from_any_boundary_match_a_compact_gate(dtype, offset, V):
    """Gate rows that start 4, 8 or 12 bytes past a 16-byte boundary (read as they lie) or on an odd element (copied first):
    the same bits as from a compact copy, forward and backward."""
    B, T, H = 2, 19, 3
    gen = torch.Generator().manual_seed(offset)
    o = torch.randn(B, T, H, V, generator=gen).to(dtype).cuda().requires_grad_(True)
    w = (1 + 0.1 * torch.randn(V, generator=gen)).to(dtype).cuda().requires_grad_(True)
    proj = torch.randn(B, T, offset + H * V, generator=gen).to(dtype).cuda()
    dy = torch.randn(B, T, H, V, generator=gen).to(dtype).cuda()
    results = []
    for gate in (proj[..., offset:], proj[..., offset:].contiguous()):
        with torch.no_grad():
            y = lm_engine_amd.gated_rmsnorm(o, gate, w, 1e-5)
        gate = gate.detach().requires_grad_(True)
        under_grad = lm_engine_amd.gated_rmsnorm(o, gate, w, 1e-5)
        results.append((y, under_grad, *torch.autograd.grad(under_grad, (o, gate, w), dy)))
    for got, want in zip(*results):
        assert torch.equal(got, want)


def test_rejected_arguments():
    o = torch.randn(2, 3, 4, 20, device="cuda")
    with pytest.raises(ValueError):
        lm_engine_amd.gated_rmsnorm(o, None, None)  # V not a multiple of 8
    with pytest.raises(ValueError):
        lm_engine_amd.gated_rmsnorm(torch.randn(2, 3, 4, 16), None, None)  # not on the GPU
    a = torch.randn(2, 5, 4, device="cuda")
    with pytest.raises(ValueError):
        lm_engine_amd.delta_rule_gates(a, a, torch.zeros(3), torch.zeros(4))


@pytest.mark.parametrize("rows,cols", [(1, 1), (63, 15), (64, 16), (65, 17), (2048, 512)])
def test_column_sums(rows, cols):
    """Two partial arrays of different widths in one launch, fp32 and bf16 results.  Each element is at most rows / 64 + 6
    rounded additions deep; bf16 adds half a unit in its eighth bit."""
    from lm_engine_amd import _lib
    from lm_engine_amd.layer_ops import column_sums

    gen = torch.Generator().manual_seed(rows + cols)
    parts = [torch.randn(rows, n, generator=gen) for n in (cols, 3 * cols + 1)]
    lib, stream = _lib.load_library(), torch.cuda.current_stream().cuda_stream
    got = column_sums(lib, stream, (parts[0].cuda(), F32), (parts[1].cuda(), BF16))
    for part, sums, unit in zip(parts, got, (0.0, 2.0**-8)):
        want = part.double().sum(dim=0)
        bound = part.abs().double().sum(dim=0) * (rows / 64 + 7) * 2.0**-24
        assert sums.shape == want.shape
        assert ((sums.double().cpu() - want).abs() <= bound + (want.abs() + bound) * unit).all()


def test_operands_on_the_host_are_refused_before_any_launch():
    """A host tensor beside device tensors raises; its address never reaches a kernel."""
    H, V = 2, 64
    a, A = torch.zeros(2, 5, H, dtype=BF16).cuda(), torch.zeros(H).cuda()
    o, z, w = torch.zeros(2, 5, H, V, dtype=BF16).cuda(), torch.zeros(2, 5, H * V, dtype=BF16), torch.ones(V, dtype=BF16)
    with pytest.raises(ValueError, match="b is on cpu"):
        lm_engine_amd.delta_rule_gates(a, a.cpu(), A, A)
    for gate, weight, name in ((z, None, "gate"), (z.view(2, 5, H, V), w.cuda(), "gate"), (z.cuda(), w, "weight"), (None, w, "weight")):
        with pytest.raises(ValueError, match=f"{name} is on cpu"):
            lm_engine_amd.gated_rmsnorm(o, gate, weight, 1e-5)
        with pytest.raises(ValueError, match=f"{name} is on cpu"):
            lm_engine_amd.gated_rmsnorm(o.clone().requires_grad_(True), gate, weight, 1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.uint8, torch.bool, torch.float32])
@pytest.mark.parametrize("B, S", [(1, 1), (1, 64), (2, 65), (6, 1500), (15, 63), (16, 64), (17, 129), (300, 7), (1024, 64), (1025, 3), (8, 8193)])
def test_padding_mask_matches_torch(dtype, B, S):
    """One launch against sum, cumsum and conversion: whole numbers, so the same values.  Rows shared by several waves, a row per wave, more
    rows than waves and than lanes, sizes that go through torch (the launch by itself there as well); also a mask that is not contiguous."""
    from lm_engine_amd.layer_ops import _MASK_BYTES, _padding_mask_kernel, padding_mask

    ways = [padding_mask] + ([_padding_mask_kernel] if dtype in _MASK_BYTES and B <= 1024 else [])
    lengths = torch.randint(0, S + 1, (B,), generator=torch.Generator().manual_seed(B + S))
    mask = (torch.arange(S)[None, :] >= S - lengths[:, None]).to(dtype).cuda()
    strided = torch.stack((mask, torch.zeros_like(mask)), dim=-1)[..., 0]
    for x in (mask, strided, mask[:1].expand(B, S)):
        for out_dtype, way in [(o, w) for o in (torch.bfloat16, torch.float32) for w in ways]:
            got, prefix = way(x, out_dtype)
            assert torch.equal(got.to(out_dtype), x.to(out_dtype))
            assert prefix.dtype == torch.int32
            assert torch.equal(prefix.cpu(), torch.nn.functional.pad(x.cpu().long().sum(-1).cumsum(0), (1, 0)).int())
