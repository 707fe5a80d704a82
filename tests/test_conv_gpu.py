"""Parity of the depthwise causal convolution kernel (through the C ABI) against the CPU oracle,
in the three modes of the reference module and with the properties its own tests assert
(tests/depthwise_causal_convolution_test.py of the reference).

Gates: fp32 within 1e-5 (the tolerance the reference's tests use); bf16 within max-abs 2e-2 and
relative-L2 1e-2 of the fp64 oracle on the same rounded inputs."""

import pytest
import torch

import lm_engine_amd
from oracle.conv_oracle import depthwise_causal_convolution_ref as conv_ref
from tests.helpers import max_abs, rel_l2


pytestmark = pytest.mark.gpu
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64


def _inputs(B, S, C, ks, dtype, seed, bias=True, state=False, mask=False):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(B, S, C, generator=g).to(dtype)
    w = (torch.randn(C, 1, ks, generator=g) * 0.5).to(dtype)
    b = (torch.randn(C, generator=g) * 0.1).to(dtype) if bias else None
    st = torch.randn(B, C, ks - 1, generator=g).to(dtype) if state else None
    m = None
    if mask:
        m = torch.ones(B, S)
        for i in range(B):
            m[i, : (3 * i + 1) % max(S, 1)] = 0  # left padding of different lengths
        m = m.to(dtype)
    return x, w, b, st, m


def _check(x, w, b, st, m, activation, label):
    print(f"case: conv {label} x={tuple(x.shape)} {x.dtype} ks={w.size(-1)} bias={b is not None} "
          f"state={st is not None} mask={m is not None} act={activation}", flush=True)  # fmt: skip
    up = lambda t: None if t is None else t.to(F64)  # noqa: E731
    y_ref, s_ref = conv_ref(up(x), up(w), up(b), up(st), up(m), output_state=True, activation=activation)
    dev = lambda t: None if t is None else t.cuda()  # noqa: E731
    y, s = lm_engine_amd.depthwise_causal_convolution(dev(x), dev(w), dev(b), dev(st), dev(m), output_state=True,
                                                      activation=activation)  # fmt: skip
    torch.cuda.synchronize()
    assert y.dtype == x.dtype and s.dtype == x.dtype and tuple(s.shape) == (x.size(0), x.size(2), w.size(-1) - 1)
    y, s = y.cpu().to(F64), s.cpu().to(F64)
    print(f"   y: max-abs {max_abs(y, y_ref):.3e} rel-L2 {rel_l2(y, y_ref):.3e}   state: max-abs {max_abs(s, s_ref):.3e}", flush=True)
    if x.dtype == F32:
        torch.testing.assert_close(y, y_ref, rtol=1e-5, atol=1e-5)
    else:
        assert max_abs(y, y_ref) <= 2e-2 * max(1.0, float(y_ref.abs().max())) and rel_l2(y, y_ref) <= 1e-2
    assert torch.equal(s, s_ref)  # the state is a copy of (masked) inputs
    return y, s


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("ks", [2, 3, 4])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("activation", [None, "silu"])
def test_fresh_prefill(dtype, ks, bias, activation):
    x, w, b, st, m = _inputs(2, 70, 64, ks, dtype, seed=ks, bias=bias)
    _check(x, w, b, st, m, activation, "prefill")


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("S", [1, 2, 3, 4, 33])
def test_continuation_from_a_state(dtype, S):
    x, w, b, st, m = _inputs(3, S, 32, 4, dtype, seed=10 + S, state=True)
    _check(x, w, b, st, m, "silu", f"continuation S={S}")


@pytest.mark.parametrize("S", [1, 2, 4])
def test_zero_state_matches_fresh_prefill(S):
    x, w, b, _, _ = _inputs(2, S, 8, 4, F32, seed=20 + S)
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    y0, s0 = lm_engine_amd.depthwise_causal_convolution(xd, wd, bd, None, None, True)
    y1, s1 = lm_engine_amd.depthwise_causal_convolution(xd, wd, bd, torch.zeros(2, 8, 3, device="cuda"), None, True)
    assert torch.equal(y0, y1) and torch.equal(s0, s1)


@pytest.mark.parametrize("continuation_len", [1, 2, 4])
@pytest.mark.parametrize("n_gen_steps", [1, 2])
@pytest.mark.parametrize("prefill_len", [3, 6, 100])
def test_prefill_continuation_and_steps_match_full_sequence(continuation_len, n_gen_steps, prefill_len):
    total = prefill_len + continuation_len + n_gen_steps
    x, w, b, _, _ = _inputs(2, total, 16, 4, F32, seed=30 + total)
    x, w, b = x.cuda(), w.cuda(), b.cuda()
    conv = lm_engine_amd.depthwise_causal_convolution
    y_full, s_full = conv(x, w, b, None, None, True)
    _, st = conv(x[:, :prefill_len], w, b, None, None, True)
    y_c, st = conv(x[:, prefill_len : prefill_len + continuation_len], w, b, st, None, True)
    torch.testing.assert_close(y_c, y_full[:, prefill_len : prefill_len + continuation_len], rtol=1e-5, atol=1e-5)
    for step in range(n_gen_steps):
        at = prefill_len + continuation_len + step
        last = step == n_gen_steps - 1
        y_s, st_next = conv(x[:, at : at + 1], w, b, st, None, not last)
        torch.testing.assert_close(y_s, y_full[:, at : at + 1], rtol=1e-5, atol=1e-5)
        st = st_next if not last else st
    assert st_next is None
    _, st = conv(x[:, :prefill_len], w, b, None, None, True)
    _, st = conv(x[:, prefill_len:], w, b, st, None, True)
    assert torch.equal(st, s_full)


def test_attention_mask():
    x, w, b, st, m = _inputs(3, 40, 32, 4, BF16, seed=40, mask=True)
    y, _ = _check(x, w, b, st, m, None, "mask")
    assert torch.all(y[1, :4] == 0) and torch.all(y[2, :7] == 0)
    # all ones is a no-op
    y0, _ = lm_engine_amd.depthwise_causal_convolution(x.cuda(), w.cuda(), b.cuda(), None, None, False, None)
    y1, _ = lm_engine_amd.depthwise_causal_convolution(x.cuda(), w.cuda(), b.cuda(), None, torch.ones(3, 40, device="cuda", dtype=BF16), False, None)
    assert torch.equal(y0, y1)


def test_strided_input_rows_and_the_layer_shape():
    # the layer convolves the fused q | k | v projection: C = 2 * key_dim + value_dim; here it is a slice of a wider buffer
    B, S, C = 2, 300, 2 * 256 + 512
    x, w, b, _, _ = _inputs(B, S, C + 64, 4, BF16, seed=50)
    xs = x[:, :, 32 : 32 + C]
    ws, bs = w[32 : 32 + C], b[32 : 32 + C]
    up = lambda t: t.to(F64)  # noqa: E731
    y_ref, _ = conv_ref(up(xs), up(ws), up(bs))
    y, _ = lm_engine_amd.depthwise_causal_convolution(x.cuda()[:, :, 32 : 32 + C], ws.cuda(), bs.cuda())
    assert rel_l2(y.cpu().to(F64), y_ref) <= 1e-2


def test_rejected_arguments():
    x = torch.randn(2, 8, 16, device="cuda")
    w = torch.randn(16, 1, 4, device="cuda")
    with pytest.raises(ValueError):
        lm_engine_amd.depthwise_causal_convolution(x, torch.randn(16, 1, 5, device="cuda"))
    with pytest.raises(ValueError):
        lm_engine_amd.depthwise_causal_convolution(x, w, activation="gelu")
    with pytest.raises(ValueError):
        lm_engine_amd.depthwise_causal_convolution(x, w, input_state=torch.zeros(2, 16, 2, device="cuda"))
    with pytest.raises(ValueError):
        lm_engine_amd.depthwise_causal_convolution(torch.randn(2, 8, 18, device="cuda"), torch.randn(18, 1, 4, device="cuda"))
    with pytest.raises(ValueError):
        lm_engine_amd.depthwise_causal_convolution(x.cpu(), w.cpu())


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("masked", [False, True])
def test_long_walks_match_short_ones(dtype, masked):
    """A batch that fills the device takes longer walks, its rows one by one 4 tokens a thread: the same bits, the oracle's values."""
    x, w, b, st, m = _inputs(8, 4099, 64, 4, dtype, seed=5, state=True, mask=masked)
    y, s = _check(x, w, b, st, m, "silu", "long walks")
    for row in (0, 7):
        xr = x[row : row + 1] if m is None else x[row : row + 1] * m[row : row + 1, :, None]
        y1, s1 = lm_engine_amd.depthwise_causal_convolution(xr.cuda(), w.cuda(), b.cuda(), st[row : row + 1].cuda(), None, output_state=True)
        first = 0 if m is None else int((m[row] == 0).sum())
        assert torch.equal(y1[0, first:].cpu().to(F64), y[row, first:]) and torch.equal(s1[0].cpu().to(F64), s[row])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype, C", [(BF16, 1024), (BF16, 1544), (F32, 1028)])
@pytest.mark.parametrize("masked", [False, True])
def test_long_walks_over_several_groups_of_channels_match_short_ones(dtype, C, masked):
    """A group is 64 threads' channels, 512 in bf16 and 256 in fp32: whole ones, and a last one cut to a single thread; tokens that are no multiple of a walk's."""
    B, S = 7, 2053
    x, w, b, st, m = _inputs(B, S, C, 4, dtype, seed=C, state=True, mask=masked)
    run = lambda i, j, first=0, last=S: lm_engine_amd.depthwise_causal_convolution(  # noqa: E731
        x[i:j, first:last].cuda(), w.cuda(), b.cuda(), st[i:j].cuda(), None if m is None else m[i:j, first:last].cuda(), output_state=True)
    y, s = run(0, B)
    for i in (0, 5):  # two rows, so that a mask counts: 2 x 330 tokens are walked four at a time
        y1, _ = run(i, i + 2, 0, 330)
        assert torch.equal(y[i : i + 2, :330], y1)
    carried = x[5:, S - 203 : S - 200].transpose(1, 2).contiguous()  # (no padding that late)
    tail = _check(x[5:, S - 200 :], w, b, carried, None if m is None else m[5:, S - 200 :], "silu", f"the end of long walks, C={C}")
    assert torch.equal(tail[0], y[5:, S - 200 :].cpu().to(F64)) and torch.equal(tail[1], s[5:].cpu().to(F64))


# the state as it lies, in and out at any element, on short and on long walks, sequences shorter than the window among them
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("ks, B, S", [(2, 3, 1), (3, 3, 1), (4, 3, 1), (4, 3, 2), (3, 3, 2), (4, 3, 5), (4, 1800, 5), (3, 1800, 9)])
def test_states_at_any_element(ks, B, S, dtype):
    import ctypes

    from lm_engine_amd import _lib

    x, w, b, st, _ = (None if t is None else t.cuda() for t in _inputs(B, S, 24, ks, dtype, seed=ks + S, state=True))
    y, s = lm_engine_amd.depthwise_causal_convolution(x, w, b, st, output_state=True)
    moved, out = (torch.full((st.numel() + 2,), 7.0, dtype=dtype, device="cuda") for _ in range(2))
    moved[1:-1] = st.flatten()
    y1 = torch.empty_like(x)
    a = _lib.GdnConvArgs()
    a.x, a.weight, a.bias, a.y = x.data_ptr(), w.data_ptr(), b.data_ptr(), y1.data_ptr()
    a.input_state, a.final_state = moved[1:].data_ptr(), out[1:].data_ptr()
    a.x_stride_b, a.x_stride_s, a.y_stride_b, a.y_stride_s = S * 24, 24, S * 24, 24
    a.B, a.S, a.C, a.kernel_size, a.activation = B, S, 24, ks, _lib.GDN_ACT_SILU
    a.dtype = a.w_dtype = _lib.GDN_BF16 if dtype == BF16 else _lib.GDN_F32
    print(f"case: conv states at an odd element, {B} x {S} ks={ks} {dtype}", flush=True)
    assert _lib.load_library().gdn_causal_conv1d_fwd(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert torch.equal(y1, y) and torch.equal(out[1:-1].view(s.shape), s) and out[0] == out[-1] == 7.0


# the ends of a walk of 4 and of 8 tokens and one past each; sequences shorter than the window
@pytest.mark.parametrize("dtype, w_dtype", [(BF16, BF16), (BF16, F32), (F32, F32)])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("ks, S", [(4, 1), (4, 2), (4, 3), (3, 4), (2, 5), (4, 7), (4, 8), (3, 9), (4, 11), (4, 12), (4, 13), (2, 16), (4, 25)])
def test_walks_of_any_length_end_where_the_sequence_does(ks, S, masked, dtype, w_dtype):
    """Enough rows to fill the device take the longer walks, a few of them the short one: the same bits, the oracle's values."""
    x, w, b, st, m = _inputs(1800, S, 24, ks, dtype, seed=S + ks, state=True, mask=masked)
    w, b = w.to(w_dtype), b.to(w_dtype)
    run = lambda n: lm_engine_amd.depthwise_causal_convolution(  # noqa: E731
        x[:n].cuda(), w.cuda(), b.cuda(), st[:n].cuda(), None if m is None else m[:n].cuda(), output_state=True)
    (y, s), (y1, s1) = run(1800), run(5)
    assert torch.equal(y[:5], y1) and torch.equal(s[:5], s1)
    _check(x[:5], w, b, st[:5], None if m is None else m[:5], "silu", f"walks ks={ks} S={S}")


@pytest.mark.gpu
@pytest.mark.parametrize("C", [8, 144, 152, 512, 520])
@pytest.mark.parametrize("S", [1, 15, 16, 17, 61])
def test_mask_values_reach_every_row_of_a_partly_filled_wave(C, S):
    """A wave keeps its rows' mask values one per lane: fewer channel vectors than values (C = 8: 1 of 64 lanes, 144 and 152: 18 and 19
    for 16 + 3 values, 520: a last wave of one), mask values other than 0 and 1, both walk lengths."""
    for B in (2, 40 * 2048 // max(S, 16) if S > 16 and C <= 152 else 3):
        x, w, b, st, m = _inputs(B, S, C, 4, BF16, seed=C + S, state=True, mask=True)
        m = m * 2.0 ** (torch.arange(S) % 3 - 1)[None, :].to(m.dtype)  # (powers of two: the state is compared bit for bit)
        _check(x, w, b, st, m, "silu", f"C={C} S={S}")
