"""Gradients through the layer's single-kernel steps and through the whole chain
(convolution -> gates -> operator -> gated norm), against autograd through the fp64 CPU oracles."""

import pytest
import torch

import lm_engine_amd
from oracle import recurrent_gated_delta_rule_ref
from oracle.conv_oracle import depthwise_causal_convolution_ref
from oracle.layer_oracle import delta_rule_gates_ref, gated_rmsnorm_ref
from tests.helpers import rel_l2


pytestmark = pytest.mark.gpu
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64


def _grads(fn, tensors, cotangents):
    leaves = [x.detach().clone().requires_grad_(True) for x in tensors]
    outs = fn(*leaves)
    outs = [o for o in outs if o is not None]
    loss = sum((o.to(c.dtype) * c).sum() for o, c in zip(outs, cotangents))
    return torch.autograd.grad(loss, leaves)


def _grads_allow_unused(fn, tensors, cotangents):
    leaves = [x.detach().clone().requires_grad_(True) for x in tensors]
    outs = [o for o in fn(*leaves) if o is not None]
    loss = sum((o.to(c.dtype) * c).sum() for o, c in zip(outs, cotangents))
    return torch.autograd.grad(loss, leaves, allow_unused=True)


def _compare(got, want, tol, names):
    for name, a, b in zip(names, got, want):
        err = rel_l2(a, b)
        assert err <= tol, f"{name}: rel-L2 {err:.3e} > {tol}"


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 6e-3)])
@pytest.mark.parametrize("shape,H", [((3, 50), 8), ((2, 1031), 12), ((777,), 40)])
def test_gates_gradients(dtype, tol, shape, H):
    """The gates' backward kernel (da, db per token, dA_log and ddt_bias reduced over tokens) against autograd
    through the fp64 oracle, on the values the kernel reads (bf16 inputs are rounded first); a and b are column
    slices of one wider projection, as the layer hands them over."""
    gen = torch.Generator().manual_seed(1)
    proj = torch.randn(*shape, 2 * H + 3, generator=gen).to(dtype)
    A_log, dt_bias = torch.randn(H, generator=gen), torch.randn(H, generator=gen)
    cg, cb = torch.randn(*shape, H, generator=gen), torch.randn(*shape, H, generator=gen).to(dtype)
    cut = lambda p: (p[..., :H], p[..., H + 3 :])  # noqa: E731

    def ref(p, A, d):
        return delta_rule_gates_ref(*cut(p), A, d, True)

    def ours(p, A, d):
        return lm_engine_amd.delta_rule_gates(*cut(p), A, d, True)

    want = _grads(ref, [x.to(F64) for x in (proj, A_log, dt_bias)], [cg.to(F64), cb.to(F64)])
    got = _grads(ours, [x.cuda() for x in (proj, A_log, dt_bias)], [cg.cuda(), cb.cuda()])
    keep = torch.ones(2 * H + 3, dtype=torch.bool)
    keep[H : H + 3] = False
    assert torch.count_nonzero(got[0][..., ~keep]) == 0
    _compare([got[0][..., keep], *got[1:]], [want[0][..., keep], *want[1:]], tol, ("da|db", "dA_log", "ddt_bias"))


@pytest.mark.parametrize("H", [1, 2, 3, 5, 16, 17, 64, 65, 128, 255, 257, 300])
def test_gates_gradients_of_any_number_of_heads(H):
    # a head's sums in a workgroup are added up by 16, 8, 4, 2 threads or one, from 256 sums down to none; tolerance as above
    test_gates_gradients(torch.float32, 1e-5, (2, 1 + 1100 // H), H)


def test_gates_gradient_of_one_output_only():
    gen = torch.Generator().manual_seed(4)
    H = 16
    a, b = torch.randn(5, 33, H, generator=gen), torch.randn(5, 33, H, generator=gen)
    A_log, dt_bias = torch.randn(H, generator=gen), torch.randn(H, generator=gen)
    c = torch.randn(5, 33, H, generator=gen)
    for which in (0, 1):
        want = _grads_allow_unused(lambda *t: (delta_rule_gates_ref(*t, False)[which],), [x.to(F64) for x in (a, b, A_log, dt_bias)], [c.to(F64)])
        got = _grads_allow_unused(lambda *t: (lm_engine_amd.delta_rule_gates(*t, False)[which],), [x.cuda() for x in (a, b, A_log, dt_bias)], [c.cuda()])
        for name, x, y in zip(("da", "db", "dA_log", "ddt_bias"), got, want):
            if y is None:
                assert x is None or torch.count_nonzero(x) == 0, name
            else:
                assert rel_l2(x, y) <= 1e-5, name


@pytest.mark.parametrize("gated", [False, True])
def test_gated_rmsnorm_gradients(gated):
    gen = torch.Generator().manual_seed(2)
    o, gate, w = torch.randn(2, 40, 4, 64, generator=gen), torch.randn(2, 40, 4, 64, generator=gen), torch.randn(64, generator=gen)
    c = torch.randn(2, 40, 4, 64, generator=gen)
    if gated:
        want = _grads(lambda o, g, w: (gated_rmsnorm_ref(o, g, w, 1e-5),), [x.to(F64) for x in (o, gate, w)], [c.to(F64)])
        got = _grads(lambda o, g, w: (lm_engine_amd.gated_rmsnorm(o, g, w, 1e-5),), [x.cuda() for x in (o, gate, w)], [c.cuda()])
        _compare(got, want, 1e-5, ("do", "dgate", "dweight"))
    else:
        want = _grads(lambda o, w: (gated_rmsnorm_ref(o, None, w, 1e-5),), [x.to(F64) for x in (o, w)], [c.to(F64)])
        got = _grads(lambda o, w: (lm_engine_amd.gated_rmsnorm(o, None, w, 1e-5),), [x.cuda() for x in (o, w)], [c.cuda()])
        _compare(got, want, 1e-5, ("do", "dweight"))


@pytest.mark.parametrize("V, gated, weighted", [(128, True, True), (256, True, False), (64, False, True), (72, True, True)])
def test_gated_rmsnorm_gradients_bf16(V, gated, weighted):
    """bf16, gate as a strided slice of a wider projection: the backward is ``gdn_gated_rmsnorm_bwd``."""
    gen = torch.Generator().manual_seed(V)
    B, S, H = 2, 33, 3
    o = torch.randn(B, S, H, V, generator=gen).to(BF16)
    proj = torch.randn(B, S, 2 * H + H * V, generator=gen).to(BF16)
    w = (1 + 0.1 * torch.randn(V, generator=gen)).to(BF16)
    c = torch.randn(B, S, H, V, generator=gen).to(BF16)

    def oracle(o, proj, w):
        gate = proj[..., 2 * H :] if gated else None
        return (gated_rmsnorm_ref(o, gate, w if weighted else None, 1e-5),)

    def kernels(o, proj, w):
        gate = proj[..., 2 * H :] if gated else None
        return (lm_engine_amd.gated_rmsnorm(o, gate, w if weighted else None, 1e-5),)

    want = _grads_allow_unused(oracle, [t.to(F64) for t in (o, proj, w)], [c.to(F64)])
    got = _grads_allow_unused(kernels, [t.cuda() for t in (o, proj, w)], [c.cuda()])
    for name, a, b in zip(("do", "dproj", "dweight"), got, want):
        if b is None:
            assert a is None, name
        else:
            assert rel_l2(a, b) <= 1e-2, f"{name}: rel-L2 {rel_l2(a, b):.3e}"


@pytest.mark.parametrize("S, ks", [(1, 4), (2, 3), (64, 4), (130, 2), (200, 4)])
@pytest.mark.parametrize("with_state, masked, silu", [(False, False, True), (True, False, True), (False, True, True), (True, True, False)])
def test_convolution_gradients_bf16_kernel(with_state, masked, silu, S, ks):
    """bf16 x: the backward is ``gdn_causal_conv1d_bwd``; against autograd through the fp64 oracle on the same
    (rounded) inputs.  The gradient is taken of y only (the cache state is not differentiated through)."""
    gen = torch.Generator().manual_seed(100 * S + ks)
    B, C = 3, 72
    rt = lambda t: t.to(BF16)  # noqa: E731
    x, w = rt(torch.randn(B, S, C, generator=gen)), rt(0.5 * torch.randn(C, 1, ks, generator=gen))
    bias, state = rt(torch.randn(C, generator=gen)), rt(torch.randn(B, C, ks - 1, generator=gen))
    cy = rt(torch.randn(B, S, C, generator=gen))
    mask = torch.ones(B, S)
    if masked and S > 1:
        mask[1, : S // 3] = 0
        mask[2, : S - 1] = 0
    m = mask if masked else None
    act = "silu" if silu else None
    tensors = [x, w, bias] + ([state] if with_state else [])
    oracle = lambda x, w, b, s=None: (depthwise_causal_convolution_ref(x, w, b, s, m, False, act)[0],)  # noqa: E731
    kernels = lambda x, w, b, s=None: (lm_engine_amd.depthwise_causal_convolution(  # noqa: E731
        x, w, b, s, None if m is None else m.cuda(), True, act)[0],)  # fmt: skip
    want = _grads(oracle, [t.to(F64) for t in tensors], [cy.to(F64)])
    got = _grads(kernels, [t.cuda() for t in tensors], [cy.cuda()])
    assert [g.dtype for g in got] == [t.dtype for t in tensors]
    names = ("dx", "dweight", "dbias", "dstate")
    for name, a, b in zip(names, got, want):
        if float(b.abs().max()) == 0.0:
            assert not a.any(), name
        else:
            assert rel_l2(a, b) <= 1e-2, f"{name}: rel-L2 {rel_l2(a, b):.3e}"


@pytest.mark.parametrize("S, ks", [(37, 4), (1, 4), (2, 3), (200, 2)])
@pytest.mark.parametrize("with_state, masked", [(False, False), (True, False), (False, True), (True, True)])
def test_convolution_gradients(with_state, masked, S, ks):
    """fp32 x: ``gdn_causal_conv1d_bwd`` again (4 channels per 16-byte access), and the gradient that flows into the
    returned state (rows of dx, or of dstate when the sequence is shorter than the state)."""
    gen = torch.Generator().manual_seed(3)
    B, C = 3, 68
    x, w, bias = torch.randn(B, S, C, generator=gen), 0.5 * torch.randn(C, 1, ks, generator=gen), torch.randn(C, generator=gen)
    state = torch.randn(B, C, ks - 1, generator=gen)
    mask = torch.ones(B, S)
    if masked and S > 1:
        mask[1, : S // 3] = 0
        mask[2, : S - 1] = 0
    cy, cs = torch.randn(B, S, C, generator=gen), torch.randn(B, C, ks - 1, generator=gen)
    m = mask if masked else None
    if with_state:
        want = _grads(lambda x, w, b, s: depthwise_causal_convolution_ref(x, w, b, s, m, True), [t.to(F64) for t in (x, w, bias, state)], [cy.to(F64), cs.to(F64)])
        got = _grads(lambda x, w, b, s: lm_engine_amd.depthwise_causal_convolution(x, w, b, s, None if m is None else m.cuda(), True),
                     [t.cuda() for t in (x, w, bias, state)], [cy.cuda(), cs.cuda()])  # fmt: skip
        _compare(got, want, 1e-5, ("dx", "dweight", "dbias", "dstate"))
    else:
        want = _grads(lambda x, w, b: depthwise_causal_convolution_ref(x, w, b, None, m, True), [t.to(F64) for t in (x, w, bias)], [cy.to(F64), cs.to(F64)])
        got = _grads(lambda x, w, b: lm_engine_amd.depthwise_causal_convolution(x, w, b, None, None if m is None else m.cuda(), True),
                     [t.cuda() for t in (x, w, bias)], [cy.cuda(), cs.cuda()])  # fmt: skip
        _compare(got, want, 1e-5, ("dx", "dweight", "dbias"))


@pytest.mark.parametrize("B, S, C", [(2, 193, 516), (16, 4097, 8), (32, 4097, 8), (1, 257, 1028)])
def test_convolution_gradients_in_every_block_length(B, S, C):
    """The walk of ``gdn_causal_conv1d_bwd`` in blocks of 64, 128 and 256 tokens (the launch picks by the workgroups it gives), the last
    block of a row one token long, channels in one workgroup and a few past it.  fp32: sums of up to 256 terms in a block and of the
    blocks, 2^-24 per addition and a growth with the root of their number, stay under 2e-6 of the result; 1e-5 as above."""
    from lm_engine_amd.conv import _backward_tokens_per_block

    assert _backward_tokens_per_block(B, S, C) == {16: 128, 32: 256}.get(B, 64)
    gen = torch.Generator().manual_seed(S + C)
    x, w, bias = torch.randn(B, S, C, generator=gen), 0.5 * torch.randn(C, 1, 4, generator=gen), torch.randn(C, generator=gen)
    cy = torch.randn(B, S, C, generator=gen)
    want = _grads(lambda x, w, b: depthwise_causal_convolution_ref(x, w, b, None, None, False, "silu")[:1], [t.to(F64) for t in (x, w, bias)], [cy.to(F64)])
    got = _grads(lambda x, w, b: lm_engine_amd.depthwise_causal_convolution(x, w, b, None, None, True, "silu")[:1],
                 [t.cuda() for t in (x, w, bias)], [cy.cuda()])  # fmt: skip
    _compare(got, want, 1e-5, ("dx", "dweight", "dbias"))


def test_layer_chain_gradients():
    B, S, HK, HV, DK, DV = 2, 130, 2, 4, 128, 128
    key_dim, value_dim = HK * DK, HV * DV
    gen = torch.Generator().manual_seed(4)
    qkv = torch.randn(B, S, 2 * key_dim + value_dim, generator=gen).to(BF16)
    ab = torch.randn(B, S, 2 * HV + value_dim, generator=gen).to(BF16)
    conv_w = (0.4 * torch.randn(2 * key_dim + value_dim, 1, 4, generator=gen)).to(BF16)
    conv_b = (0.1 * torch.randn(2 * key_dim + value_dim, generator=gen)).to(BF16)
    A_log = torch.log(torch.rand(HV, generator=gen) * 4 + 0.1)
    dt_bias = torch.randn(HV, generator=gen) - 2.0
    norm_w = (1 + 0.1 * torch.randn(DV, generator=gen)).to(BF16)
    c = torch.randn(B, S, value_dim, generator=gen)

    def oracle(qkv, ab, conv_w, conv_b, A_log, dt_bias, norm_w):
        y, _ = depthwise_causal_convolution_ref(qkv, conv_w, conv_b, None, None, False)
        q, k, v = y.split((key_dim, key_dim, value_dim), dim=-1)
        q = q.reshape(B, S, HK, DK).repeat_interleave(HV // HK, dim=-2)
        k = k.reshape(B, S, HK, DK).repeat_interleave(HV // HK, dim=-2)
        v = v.reshape(B, S, HV, DV)
        a, b, gate = ab[..., :HV], ab[..., HV : 2 * HV], ab[..., 2 * HV :]
        g, beta = delta_rule_gates_ref(a, b, A_log, dt_bias, False)
        o, _ = recurrent_gated_delta_rule_ref(q, k, v, g=g, beta=beta, use_qk_l2norm_in_kernel=True, state_dtype=F64)
        return (gated_rmsnorm_ref(o, gate, norm_w, 1e-5).flatten(-2),)

    def kernels(qkv, ab, conv_w, conv_b, A_log, dt_bias, norm_w):
        a, b, gate = ab[..., :HV], ab[..., HV : 2 * HV], ab[..., 2 * HV :]
        out, _ = lm_engine_amd.gated_deltanet_mixing(qkv, a, b, gate, conv_w, conv_b, A_log, dt_bias, norm_w, 1e-5,
                                                     HK, HV, DK, DV)  # fmt: skip
        return (out,)

    tensors = (qkv, ab, conv_w, conv_b, A_log, dt_bias, norm_w)
    want = _grads(oracle, [t.to(F64) for t in tensors], [c.to(F64)])
    got = _grads(kernels, [t.cuda() for t in tensors], [c.cuda()])
    assert [g.dtype for g in got] == [t.dtype for t in tensors]
    _compare(got, want, 3e-2, ("dqkv", "dab", "dconv_weight", "dconv_bias", "dA_log", "ddt_bias", "dnorm_weight"))


@pytest.mark.parametrize("B, S, HK, H, K, V", [(2, 192, 2, 2, 128, 64), (1, 130, 3, 3, 64, 64), (2, 128, 2, 4, 64, 64), (1, 64, 2, 2, 256, 512)])
def test_gradients_of_column_blocks_are_those_of_separate_tensors(B, S, HK, H, K, V):
    """q, k and v as column blocks of one tensor get gradients that are column blocks of one (written with its token stride);
    the values are those of three separate tensors, bit for bit (every sum of the kernels has one order), and the layer's split hands
    them on without a copy."""
    from lm_engine_amd.layer import _SplitChannels
    from lm_engine_amd.ops import column_blocks

    gen = torch.Generator().manual_seed(S)
    qkv = torch.randn(B, S, 2 * HK * K + H * V, generator=gen).to(torch.bfloat16).cuda().requires_grad_(True)
    g = -torch.rand(B, S, H, generator=gen).cuda()
    beta = torch.rand(B, S, H, generator=gen).to(torch.bfloat16).cuda()
    d_o = torch.randn(B, S, H, V, generator=gen).to(torch.bfloat16).cuda()
    blocks = _SplitChannels.apply(qkv, HK, H, K, V)
    separate = [x.detach().contiguous().requires_grad_(True) for x in blocks]
    assert column_blocks(*blocks) and not column_blocks(*separate) and not column_blocks(blocks[1], blocks[0], blocks[2])

    def grads(q, k, v, wrt):
        o, _ = lm_engine_amd.chunk_gated_delta_rule(q, k, v, g, beta, use_qk_l2norm_in_kernel=True)
        return torch.autograd.grad(o, wrt, d_o, retain_graph=True)

    joined, apart = grads(*blocks, blocks), grads(*separate, separate)
    assert column_blocks(*joined) == (HK == H)
    for a, b in zip(joined, apart):
        assert torch.equal(a, b)
    (whole,) = grads(*blocks, (qkv,))
    assert torch.equal(whole, torch.cat([x.flatten(-2) for x in apart], dim=-1))
    # one of the three does not get a gradient, or gets a larger one
    (part,) = torch.autograd.grad((2 * blocks[2].float()).sum(), (qkv,), retain_graph=True)
    assert (part[..., 2 * HK * K :] == 2).all() and not part[..., : 2 * HK * K].any()


def _layouts(dense):
    """``dense`` as backward functions of other operations hand gradients on: a column block of a wider tensor (strides that are no
    multiple of 8, then odd ones) and a view that starts at an odd element."""
    for extra in (4, 1):
        wide = torch.cat([dense, torch.full((*dense.shape[:-1], extra), float("nan"), dtype=dense.dtype, device="cuda")], dim=-1)
        yield f"{extra} columns wider", wide[..., : dense.size(-1)]
    flat = torch.full((dense.numel() + 1,), float("nan"), dtype=dense.dtype, device="cuda")
    shifted = flat[1:].view(dense.shape)
    yield "at an odd element", shifted.copy_(dense)


@pytest.mark.parametrize("step", ["operator, V = 64", "operator, V = 32", "operator, fp32", "convolution", "norm", "gates"])
def test_gradients_flow_in_whatever_their_layout(step):
    """The layout of an incoming gradient is chosen by whatever consumed the output: every layout gives the gradients of the dense one,
    in the same bits (the same kernels on the same values)."""
    gen = torch.Generator().manual_seed(7)
    dtype = F32 if step.endswith("fp32") else BF16
    leaf = lambda *shape: torch.randn(*shape, generator=gen).to(dtype).cuda().requires_grad_(True)  # noqa: E731
    B, T, H, K = 2, 130, 2, 64
    V = 32 if step.endswith("32") else 64
    if step.startswith("operator"):
        q, k, v, h0 = leaf(B, T, H, K), leaf(B, T, H, K), leaf(B, T, H, V), leaf(B, H, K, V).detach().float().requires_grad_(True)
        leaves = [q, k, v, h0]
        outputs = lm_engine_amd.chunk_gated_delta_rule(q, k, v, initial_state=h0, output_final_state=True, use_qk_l2norm_in_kernel=True)
    elif step == "convolution":
        leaves = [leaf(B, T, 64), leaf(64, 4), leaf(64)]
        outputs = lm_engine_amd.depthwise_causal_convolution(*leaves)[:1]
    elif step == "norm":
        leaves = [leaf(B, T, H, V), leaf(B, T, H, V), leaf(V)]
        outputs = (lm_engine_amd.gated_rmsnorm(*leaves, 1e-5),)
    else:
        leaves = [leaf(B, T, H), leaf(B, T, H), leaf(H).detach().float().requires_grad_(True), leaf(H).detach().float().requires_grad_(True)]
        outputs = lm_engine_amd.delta_rule_gates(*leaves)
    dense = [torch.randn(o.shape, generator=gen).to(o.dtype).cuda() for o in outputs]
    want = torch.autograd.grad(outputs, leaves, dense, retain_graph=True)
    for j, d in enumerate(dense):
        for name, x in _layouts(d):
            print(f"case: {step}, gradient of output {j} {name}", flush=True)
            got = torch.autograd.grad(outputs, leaves, [*dense[:j], x, *dense[j + 1 :]], retain_graph=True)
            assert all(torch.equal(a, b) for a, b in zip(got, want)), name
