"""The native host path of the entry points (csrc/gdn_host.cpp): what it hands on to the Python code, what it raises,
and what it leaves behind.  The library's entry points are replaced by small stand-ins where a test needs a status or a look
at the thread's state: nothing is launched then."""

import contextlib
import ctypes
import sys

import pytest
import torch

import lm_engine_amd
from lm_engine_amd import _host, _lib

from .helpers import rel_l2


pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@contextlib.contextmanager
def _entry_points_replaced(**stand_ins):
    """Binds ``name=address`` in place of the library's own entry points."""
    module, lib = _host.host(), _lib.load_library()
    own = {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _host._BOUND}
    module.bind(_lib.check_status, *({**own, **stand_ins}[name] for name in _host._BOUND))
    try:
        yield
    finally:
        module.bind(_lib.check_status, *own.values())


def _layer_operands(B, S, H=2, K=64, V=64, seed=1):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *shape: torch.randn(*shape, generator=gen).to(BF16).cuda()  # noqa: E731
    C = H * (2 * K + V)
    return dict(qkv=r(B, S, C), a=r(B, S, H), b=r(B, S, H), gate=r(B, S, H * V), conv_weight=0.3 * r(C, 1, 4), conv_bias=0.1 * r(C),
                A_log=torch.zeros(H).cuda(), dt_bias=torch.zeros(H).cuda(), norm_weight=r(V), norm_eps=1e-5,
                num_k_heads=H, num_v_heads=H, k_head_dim=K, v_head_dim=V)  # fmt: skip


def _calls():
    """``name of the C entry -> a call that ends in it``."""
    x = _layer_operands(2, 1)
    gen = torch.Generator().manual_seed(2)
    r = lambda *shape: torch.randn(*shape, generator=gen).to(BF16).cuda()  # noqa: E731
    q, k, v, long = r(2, 1, 2, 64), r(2, 1, 2, 64), r(2, 1, 2, 64), r(1, 130, 2, 64)
    h = torch.zeros(2, 2, 64, 64).cuda()
    return {
        "gdn_layer_step": lambda: lm_engine_amd.gated_deltanet_mixing(**x, cache=(None, None)),
        "gdn_causal_conv1d_fwd": lambda: lm_engine_amd.depthwise_causal_convolution(x["qkv"], x["conv_weight"], x["conv_bias"]),
        "gdn_gates_fwd": lambda: lm_engine_amd.delta_rule_gates(x["a"], x["b"], x["A_log"], x["dt_bias"]),
        "gdn_gated_rmsnorm_fwd": lambda: lm_engine_amd.gated_rmsnorm(v, None, x["norm_weight"], 1e-5),
        "gdn_recurrent_fwd": lambda: lm_engine_amd.fused_recurrent_gated_delta_rule(q, k, v, initial_state=h, output_final_state=True,
                                                                                      inplace_state=True),
        "gdn_chunk_fwd": lambda: lm_engine_amd.chunk_gated_delta_rule(long, long, long),
    }  # fmt: skip


@pytest.mark.parametrize("entry", ["gdn_layer_step", "gdn_causal_conv1d_fwd", "gdn_gates_fwd", "gdn_gated_rmsnorm_fwd", "gdn_recurrent_fwd",
                                   "gdn_chunk_fwd"])  # fmt: skip
def test_a_hip_error_is_raised_and_the_call_not_made_again(entry):
    """A positive status can come with a launch that is in the stream (the error was pending on the thread): a second launch
    of an in-place step would advance its state twice.  A negative one (nothing launched) goes to the Python path."""
    made = []

    def stand_in(status):
        @ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p)
        def fn(args, stream):
            made.append(status)
            return status

        return fn

    call = _calls()[entry]
    call()
    failing, refusing = stand_in(1), stand_in(-3)
    with _entry_points_replaced(**{entry: ctypes.cast(failing, ctypes.c_void_p).value}):
        with pytest.raises(RuntimeError, match=f"{entry}.*status 1"):
            call()
    with _entry_points_replaced(**{entry: ctypes.cast(refusing, ctypes.c_void_p).value}):
        call()
    assert made == [1, -3]
    torch.cuda.synchronize()


@pytest.mark.parametrize("tokens", [2, 3])
def test_a_gate_of_several_tokens_beside_one_token_is_refused(tokens):
    x = _layer_operands(2, 1)
    gate = torch.randn(2, tokens, 128, generator=torch.Generator().manual_seed(3)).to(BF16).cuda()
    with pytest.raises(ValueError, match="gate must have"):
        lm_engine_amd.gated_deltanet_mixing(**{**x, "gate": gate}, cache=(None, None))


@pytest.mark.parametrize("shape", [(2, 5, 1), (2, 5, 384), (2, 4), (3, 5)])
def test_an_attention_mask_that_is_not_one_value_per_token_is_refused(shape):
    x = _layer_operands(2, 5)
    with pytest.raises(ValueError, match="attention_mask must be"):
        lm_engine_amd.depthwise_causal_convolution(x["qkv"], x["conv_weight"], attention_mask=torch.zeros(shape).cuda())


def test_a_convolution_weight_of_another_layout_is_refused():
    """``[C, 1, ks]`` and ``[C, ks]`` are what is taken, on one token (the layer's step) and on several."""
    x = _layer_operands(2, 1)
    for shape in ((384, 1, 1, 4), (384, 2, 2), (384, 4, 1)):
        weight = x["conv_weight"].reshape(shape)
        with pytest.raises(ValueError, match="weight must be|kernel_size"):
            lm_engine_amd.depthwise_causal_convolution(x["qkv"], weight)
        with pytest.raises(ValueError, match="weight must be|kernel_size"):
            lm_engine_amd.gated_deltanet_mixing(**{**x, "conv_weight": weight}, cache=(None, None))
    taken = [lm_engine_amd.gated_deltanet_mixing(**{**x, "conv_weight": x["conv_weight"].reshape(shape)}, cache=(None, None))[0]
             for shape in ((384, 1, 4), (384, 4))]  # fmt: skip
    assert torch.equal(*taken)


def test_a_step_that_ends_early_gives_its_workspace_back():
    """Several workgroups per head: the tickets' memory is asked for, then an operand turns out not to be a number."""
    x = _layer_operands(2, 1, K=128, V=256)
    owner = torch.zeros(1 << 16, dtype=torch.int32).cuda()
    before = sys.getrefcount(owner)
    result = _host.host().layer_step(
        _host.raw_stream(0), x["qkv"], x["a"], x["b"], x["gate"], x["conv_weight"], x["conv_bias"], x["A_log"], x["dt_bias"],
        x["norm_weight"], 1e-5, 2, 2, 128, 256, None, None, "not a number", 1.0, 1,
        lambda pairs, V: (owner, owner.data_ptr(), owner.data_ptr() + 4 * pairs))  # fmt: skip
    assert result is None and sys.getrefcount(owner) == before


@pytest.mark.parametrize("entry", ["gdn_layer_step", "gdn_causal_conv1d_fwd", "gdn_gates_fwd", "gdn_gated_rmsnorm_fwd", "gdn_recurrent_fwd",
                                   "gdn_chunk_fwd"])  # fmt: skip
def test_other_threads_run_while_a_call_launches(entry):
    """The interpreter lock is free inside the library: its own question "does this thread hold it" stands in for the entry
    point, and answers with the status 0."""
    call = _calls()[entry]
    call()
    with _entry_points_replaced(**{entry: ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value}):
        call()
    torch.cuda.synchronize()


def test_layouts_that_the_convolution_refuses_are_refused_on_one_token_too():
    """Rows off 16-byte boundaries or on top of each other: the convolution raises for them, alone and as part of the layer's step."""
    x = _layer_operands(2, 1)
    r = lambda *shape: torch.randn(*shape, generator=torch.Generator().manual_seed(5)).to(BF16).cuda()  # noqa: E731
    wide, flat = r(2, 1, 400), r(384 * 4 + 1)
    for over in (dict(qkv=wide[..., 1:385]), dict(qkv=r(2, 1, 388)[..., :384]), dict(qkv=r(384).as_strided((2, 1, 384), (0, 8, 1))), dict(conv_weight=flat[1:].view(384, 1, 4)),
                 dict(conv_bias=flat[1:385])):  # fmt: skip
        operands = {**x, **over}
        with pytest.raises(ValueError, match="gdn_causal_conv1d_fwd"):
            lm_engine_amd.depthwise_causal_convolution(operands["qkv"], operands["conv_weight"], operands["conv_bias"])
        with pytest.raises(ValueError, match="gdn_causal_conv1d_fwd"):
            lm_engine_amd.gated_deltanet_mixing(**operands, cache=(None, None))
    with pytest.raises(ValueError, match="gdn_gated_rmsnorm_fwd"):
        lm_engine_amd.gated_deltanet_mixing(**{**x, "norm_weight": flat[1:65]}, cache=(None, None))
    taken = dict(qkv=wide[..., 8:392], a=wide[..., 1:3], b=wide[..., 3:5], gate=wide[..., 7:135])  # scalars and gate lie anywhere
    out, _ = lm_engine_amd.gated_deltanet_mixing(**{**x, **taken}, cache=(None, None))
    want, _ = lm_engine_amd.gated_deltanet_mixing(**{**x, **{n: t.contiguous() for n, t in taken.items()}}, cache=(None, None))
    assert torch.equal(out, want)


class _NativePath:
    """The native host path with a record of which calls it took on; ``on`` False: it takes none."""

    def __init__(self, on):
        self.on, self.took = on, []

    def __getattr__(self, name):
        def call(*args):
            result = getattr(_host.host(), name)(*args) if self.on else None
            self.took.append(result is not None)
            return result

        return call


def _outcome(call):
    """What a call gives: its tensors, or the type and text of what it raises."""
    try:
        with torch.no_grad():
            result = call()
    except (ValueError, RuntimeError, TypeError, IndexError, AttributeError) as error:
        return type(error), str(error)
    flat = []
    for x in result if isinstance(result, tuple) else (result,):
        flat += x if isinstance(x, tuple) else (x,)
    return flat


def _operand_forms():
    """Calls in forms that a caller may use or get wrong: layouts, types, shapes, options."""
    gen = torch.Generator().manual_seed(7)
    r = lambda *shape: torch.randn(*shape, generator=gen).to(BF16).cuda()  # noqa: E731
    x3, w, bias, state = r(2, 5, 384), 0.3 * r(384, 1, 4), 0.1 * r(384), r(2, 384, 3)
    mask = (torch.rand(2, 5, generator=gen) > 0.3).cuda()
    conv = lambda *args, **kw: lambda: lm_engine_amd.depthwise_causal_convolution(*args, output_state=True, **kw)  # noqa: E731
    wide = r(2, 5, 400)
    yield "conv", {
        "plain": conv(x3, w, bias, state), "no state": conv(x3, w, bias), "no bias": conv(x3, w), "one token": conv(x3[:, :1], w, bias, state),
        "slice": conv(wide[..., 8:392], w, bias, state), "slice off its boundary": conv(wide[..., 1:385], w, bias, state),
        "tokens first": conv(r(5, 2, 384).transpose(0, 1), w, bias, state), "channels strided": conv(r(2, 384, 5).transpose(1, 2), w, bias, state),
        "fp32 weight": conv(x3, w.float(), bias.float(), state), "fp32 x": conv(x3.float(), w, bias, state), "mixed bias": conv(x3, w, bias.float()),
        "fp16": conv(x3.half(), w.half()), "state fp32": conv(x3, w, bias, state.float()), "state of another size": conv(x3, w, bias, state[..., :2]),
        "state strided": conv(x3, w, bias, r(2, 3, 384).transpose(1, 2)), "weight strided": conv(x3, r(4, 384).t(), bias), "weight 2-D": conv(x3, w[:, 0], bias),
        "weight of other channels": conv(x3, w[:383], bias), "five taps": conv(x3, r(384, 1, 5)), "one tap": conv(x3, r(384, 1, 1)), "bias 2-D": conv(x3, w, bias[None]),
        "2-D x": conv(x3[0], w), "no tokens": conv(x3[:, :0], w), "odd channels": conv(r(2, 5, 381), r(381, 1, 4)), "mask bool": conv(x3, w, bias, state, mask),
        "mask int": conv(x3, w, bias, state, mask.long()), "mask fp32": conv(x3, w, bias, state, mask.float()), "mask of one row": conv(x3, w, bias, state, mask[:1]),
        "mask of one token": conv(x3, w, bias, state, mask[:, :1]), "mask 1-D": conv(x3, w, bias, state, mask[0]), "mask 3-D of one row": conv(x3, w, bias, state, mask[:1, :, None]),
        "mask of other tokens": conv(x3, w, bias, state, mask[:, :4]), "mask on the host": conv(x3, w, bias, state, mask.cpu()), "swish": conv(x3, w, activation="swish"),
        "no activation": conv(x3, w, activation=None), "gelu": conv(x3, w, activation="gelu"), "weight on the host": conv(x3, w.cpu()),
    }  # fmt: skip
    a, b, A, dt = r(2, 5, 3), r(2, 5, 3), torch.rand(3, generator=gen).cuda(), torch.rand(3, generator=gen).cuda()
    gates = lambda *args, **kw: lambda: lm_engine_amd.delta_rule_gates(*args, **kw)  # noqa: E731
    ab = r(2, 5, 8)
    yield "gates", {
        "plain": gates(a, b, A, dt), "negative eigenvalues": gates(a, b, A, dt, allow_neg_eigval=True), "slices": gates(ab[..., :3], ab[..., 3:6], A, dt),
        "slices of one token": gates(ab[:, :1, :3], ab[:, :1, 3:6], A, dt), "every second row": gates(ab[:, ::2, :3], ab[:, ::2, 3:6], A, dt),
        "heads strided": gates(ab[..., ::3], ab[..., 1::3][..., :3], A, dt), "transposed": gates(r(5, 2, 3).transpose(0, 1), b, A, dt), "2-D": gates(a[0], b[0], A, dt),
        "1-D": gates(a[0, 0], b[0, 0], A, dt), "bf16 parameters": gates(a, b, A.to(BF16), dt.to(BF16)), "parameters 2-D": gates(a, b, A[None], dt[None]),
        "fp32": gates(a.float(), b.float(), A, dt), "mixed": gates(a, b.float(), A, dt), "other shape": gates(a, b[:, :4], A, dt), "other heads": gates(a, b, A[:2], dt),
        "no tokens": gates(a[:, :0], b[:, :0], A, dt), "parameters on the host": gates(a, b, A.cpu(), dt.cpu()), "parameters strided": gates(a, b, torch.rand(6).cuda()[::2], dt),
        "one head": gates(r(2, 5, 1), r(2, 5, 1), A[:1], dt[:1]), "b on the host": gates(a, b.cpu(), A, dt),
    }  # fmt: skip
    o, z, nw = r(2, 5, 2, 64), r(2, 5, 128), r(64)
    norm = lambda *args: lambda: lm_engine_amd.gated_rmsnorm(*args)  # noqa: E731
    zw = r(2, 5, 140)
    yield "norm", {
        "plain": norm(o, z, nw, 1e-5), "no gate": norm(o, None, nw, 1e-5), "no weight": norm(o, z, None, 1e-5), "default eps": norm(o, z, nw), "gate by heads": norm(o, z.view(2, 5, 2, 64), nw, 1e-5),
        "gate slice": norm(o, zw[..., 4:132], nw, 1e-5), "gate slice off its boundary": norm(o, zw[..., 3:131], nw, 1e-5), "gate heads strided": norm(o, r(2, 5, 64, 2).transpose(2, 3), nw, 1e-5),
        "gate of other leading dims": norm(o, z.view(10, 128), nw, 1e-5), "gate tokens first": norm(o, r(5, 2, 128).transpose(0, 1), nw, 1e-5), "gate of one token": norm(o, z[:, :1], nw, 1e-5),
        "gate fp32": norm(o, z.float(), nw, 1e-5), "o strided": norm(r(2, 2, 5, 64).transpose(1, 2), z, nw, 1e-5), "o 2-D": norm(o[0, 0], z[0, 0], nw, 1e-5), "o 2-D, gate 2-D": norm(o[0, 0], z[0, 0].view(2, 64), nw, 1e-5),
        "o 1-D": norm(o[0, 0, 0], None, nw, 1e-5), "weight fp32": norm(o, z, nw.float(), 1e-5), "weight of another size": norm(o, z, nw[:32], 1e-5), "weight 2-D": norm(o, z, nw[None], 1e-5),
        "weight strided": norm(o, z, r(128)[::2], 1e-5), "fp32": norm(o.float(), z.float(), nw.float(), 1e-5), "fp16": norm(o.half(), None, None, 1e-5), "no tokens": norm(o[:, :0], z[:, :0], nw, 1e-5),
        "odd V": norm(r(2, 5, 2, 20), None, None, 1e-5), "wide V": norm(r(2, 5, 2, 520), None, None, 1e-5), "one head": norm(r(2, 5, 1, 64), r(2, 5, 64), nw, 1e-5), "gate on the host": norm(o, z.cpu(), nw, 1e-5),
    }  # fmt: skip
    for T, op in ((5, lm_engine_amd.fused_recurrent_gated_delta_rule), (130, lm_engine_amd.chunk_gated_delta_rule)):
        q, k, v = r(2, T, 2, 64), r(2, T, 2, 64), r(2, T, 4, 64)
        g, beta, h = -torch.rand(2, T, 4, generator=gen).cuda(), torch.rand(2, T, 4, generator=gen).to(BF16).cuda(), torch.randn(2, 4, 64, 64, generator=gen).cuda()
        row = lambda *xs: [x[:1] for x in xs]  # noqa: E731
        prefix = lambda *ends, dtype=torch.int32: torch.tensor(ends, dtype=dtype).cuda()  # noqa: E731
        base = dict(q=q, k=k, v=v, g=g, beta=beta, initial_state=h, output_final_state=True, use_qk_l2norm_in_kernel=True)
        packed = {**base, **dict(zip(("q", "k", "v", "g", "beta"), row(q, k, v, g, beta))), "cu_seqlens": prefix(0, 3, T)}
        padded = {**base, "left_padded": True, "cu_seqlens": prefix(0, 2, T + 2)}
        qkv = r(2, T, 2 * 64 + 2 * 64 + 4 * 64 + 8)
        views = dict(q=qkv[..., :128].view(2, T, 2, 64), k=qkv[..., 128:256].view(2, T, 2, 64), v=qkv[..., 256:512].view(2, T, 4, 64))
        off = dict(q=qkv[..., 4:132].unflatten(-1, (2, 64)))
        call = lambda over, base=base, op=op: lambda: op(**{**base, **over})  # noqa: E731
        forms = {
            "plain": call({}), "no state": call(dict(initial_state=None)), "no final state": call(dict(output_final_state=False)), "ungated": call(dict(g=None, beta=None)),
            "scale": call(dict(scale=0.3)), "scale as tensor": call(dict(scale=torch.tensor(0.3))), "no l2norm": call(dict(use_qk_l2norm_in_kernel=False)), "slices": call(views),
            "slice off its boundary": call(off), "tokens first": call(dict(q=r(T, 2, 2, 64).transpose(0, 1))), "last dim strided": call(dict(v=r(2, T, 64, 4).transpose(2, 3))),
            "equal heads": call(dict(q=r(2, T, 4, 64), k=r(2, T, 4, 64))), "heads that do not divide": call(dict(q=r(2, T, 3, 64), k=r(2, T, 3, 64))), "k of other heads": call(dict(k=r(2, T, 4, 64))),
            "g bf16": call(dict(g=g.to(BF16))), "g strided": call(dict(g=-torch.rand(2, 4, T, generator=gen).cuda().transpose(1, 2))), "g of other heads": call(dict(g=g[..., :2])), "beta fp32": call(dict(beta=beta.float())),
            "beta fp16": call(dict(beta=beta.half())), "beta 4-D": call(dict(beta=beta[..., None])), "state bf16": call(dict(initial_state=h.to(BF16))), "state of another batch": call(dict(initial_state=h[:1])),
            "state strided": call(dict(initial_state=h.transpose(2, 3))), "mixed types": call(dict(k=k.float())), "fp32": call(dict(q=q.float(), k=k.float(), v=v.float())), "fp16": call(dict(q=q.half(), k=k.half(), v=v.half())),
            "K = 96": call(dict(q=r(2, T, 2, 96), k=r(2, T, 2, 96), initial_state=None)), "V = 40": call(dict(v=r(2, T, 4, 40), initial_state=None)), "other tokens": call(dict(v=v[:, 1:])), "k on the host": call(dict(k=k.cpu())),
            "packed": call(packed), "packed, int64 prefix": call({**packed, "cu_seqlens": prefix(0, 3, T, dtype=torch.int64)}), "packed, strided prefix": call({**packed, "cu_seqlens": prefix(0, 0, 3, 0, T)[::2]}),
            "packed with an empty sequence": call({**packed, "cu_seqlens": prefix(0, 0, T)}), "packed, state of another count": call({**packed, "cu_seqlens": prefix(0, 1, 2, T)}),
            "prefix beside a batch": call(dict(cu_seqlens=prefix(0, 3, T))), "prefix of one": call({**packed, "cu_seqlens": prefix(0)}), "prefix 2-D": call({**packed, "cu_seqlens": prefix(0, 3, T)[None]}), "padded": call(padded),
            "padded, prefix too short": call({**padded, "cu_seqlens": prefix(0, T)}), "padded without prefix": call({**padded, "cu_seqlens": None}), "no tokens": call({n: base[n][:, :0] for n in ("q", "k", "v", "g", "beta")}),
        }  # fmt: skip
        if T == 5:  # in place on a copy that the outcome shows
            own = lambda h0=h, **over: lambda: (lambda s: (*op(**{**base, **over, "initial_state": s, "inplace_state": True}), s))(None if h0 is None else h0.clone())  # noqa: E731
            forms.update({"in place": own(), "in place without a state": own(None), "in place, strided": own(h.transpose(2, 3)), "in place, no final state": own(output_final_state=False)})
        yield ("recurrent", "chunk")[T > 64], forms
    x = _layer_operands(2, 1)
    zc, hc = r(2, 384, 3), torch.randn(2, 2, 64, 64, generator=gen).cuda()
    abz = r(2, 1, 2 + 2 + 128)
    step = lambda cache=(zc, hc), **over: lambda: lm_engine_amd.gated_deltanet_mixing(**{**x, **over}, cache=cache)  # noqa: E731
    yield "layer_step", {
        "plain": step(), "no cache yet": step((None, None)), "no convolution state": step((None, hc)), "no gate": step(gate=None), "no norm weight": step(norm_weight=None), "no bias": step(conv_bias=None),
        "slices": step(a=abz[..., :2], b=abz[..., 2:4], gate=abz[..., 4:]), "gate by heads": step(gate=r(2, 1, 2, 64)), "gate 2-D": step(gate=r(2, 128)), "gate of another batch": step(gate=r(1, 1, 128)), "gate fp32": step(gate=r(2, 1, 128).float()),
        "a of another batch": step(a=r(1, 1, 2)), "a fp32": step(a=r(2, 1, 2).float()), "bf16 decay": step(A_log=x["A_log"].to(BF16), dt_bias=x["dt_bias"].to(BF16)), "fp32 convolution weight": step(conv_weight=x["conv_weight"].float(), conv_bias=x["conv_bias"].float()),
        "fp32 norm weight": step(norm_weight=x["norm_weight"].float()), "norm weight of another size": step(norm_weight=r(32)), "state bf16": step((zc, hc.to(BF16))), "convolution state fp32": step((zc.float(), hc)), "convolution state strided": step((r(2, 3, 384).transpose(1, 2), hc)),
        "convolution state of another size": step((zc[..., :2], hc)), "state of another batch": step((zc, hc[:1])), "no activation": step(conv_activation=None), "gelu": step(conv_activation="gelu"), "negative eigenvalues": step(allow_neg_eigval=True), "scale": step(scale=0.2),
        "default eps": step(norm_eps=None), "qkv slice": step(qkv=r(2, 1, 400)[..., 8:392]), "qkv slice off its boundary": step(qkv=r(2, 1, 400)[..., 1:385]), "qkv of other channels": step(qkv=r(2, 1, 392)), "fp32": step((zc.float(), hc), **{n: y.float() for n, y in x.items() if isinstance(y, torch.Tensor)}),
        "mask": step(attention_mask=torch.ones(2, 1).cuda()), "state on the host": step((zc, hc.cpu())), "gate on the host": step(gate=r(2, 1, 128).cpu()),
    }  # fmt: skip


def test_calls_end_as_they_do_without_the_native_path(monkeypatch):
    """Every form of a call gives the same bits, or raises the same error, with the native host path and without it.  The layer's
    one-launch step adds the norm's squares up in another order (its output: an ulp; its states: the same bits)."""
    from lm_engine_amd import conv, layer, layer_ops, ops

    differ = []
    for name, forms in _operand_forms():
        for form, call in forms.items():
            print(f"case: {name}, {form}", flush=True)
            outcomes = []
            for path in (_NativePath(True), _NativePath(False)):
                with monkeypatch.context() as m:
                    for module in (conv, layer, layer_ops, ops):
                        m.setattr(module, "host", lambda path=path: path)
                    outcomes.append(_outcome(call))
                assert form != "plain" or path.took[0] == path.on, "the path under test was not the one taken"
            native, python = outcomes
            same = native == python if isinstance(native, tuple) or isinstance(python, tuple) else len(native) == len(python) and all(
                (x is None and y is None) or (x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride()
                                              and (torch.equal(x, y) or (name == "layer_step" and i == 0 and rel_l2(x, y) <= 1e-3)))
                for i, (x, y) in enumerate(zip(native, python)))  # fmt: skip
            if not same:
                differ.append((name, form, *(z if isinstance(z, tuple) else "tensors" for z in (native, python))))
    torch.cuda.synchronize()
    assert not differ, "\n".join(map(str, differ))


def _training_forms():
    """``(name of the native backward, {form: (function, operands that want a gradient)})``"""
    gen = torch.Generator().manual_seed(21)
    r = lambda *shape: torch.randn(*shape, generator=gen).to(BF16).cuda()  # noqa: E731
    x, w, bias, mask = r(2, 70, 384), 0.3 * r(384, 1, 4), 0.1 * r(384), (torch.rand(2, 70, generator=gen) > 0.3).to(BF16).cuda()
    conv = lambda **kw: lambda *t: lm_engine_amd.depthwise_causal_convolution(*t, **kw)[0]  # noqa: E731
    yield "conv_bwd", {
        "plain": (conv(), (x, w, bias)), "no bias": (conv(), (x, w)), "2-D weight": (conv(), (x, w[:, 0])), "mask": (conv(attention_mask=mask), (x, w, bias)),
        "mask int": (conv(attention_mask=mask.long()), (x, w, bias)), "mask of one row": (conv(attention_mask=mask[:1]), (x, w, bias)), "no activation": (conv(activation=None), (x, w, bias)),
        "fp32": (conv(), (x.float(), w.float(), bias.float())), "fp32 weight": (conv(), (x, w.float(), bias.float())), "slice": (conv(), (r(2, 70, 400)[..., 8:392], w, bias)),
        "state": (lambda x, w, s: lm_engine_amd.depthwise_causal_convolution(x, w, None, s)[0], (x, w, r(2, 384, 3))), "one token": (conv(), (x[:, :1], w, bias)),
    }  # fmt: skip
    a, b, A, dt, ab = r(2, 70, 3), r(2, 70, 3), torch.rand(3, generator=gen).cuda(), torch.rand(3, generator=gen).cuda(), r(2, 70, 8)
    gates = lambda *t, **kw: torch.cat([y.float().flatten() for y in lm_engine_amd.delta_rule_gates(*t, **kw)])  # noqa: E731
    yield "gates_bwd", {
        "plain": (gates, (a, b, A, dt)), "slices": (gates, (ab[..., :3], ab[..., 3:6], A, dt)), "negative eigenvalues": (lambda *t: gates(*t, allow_neg_eigval=True), (a, b, A, dt)),
        "bf16 decay": (gates, (a, b, A.to(BF16), dt.to(BF16))), "fp32": (gates, (a.float(), b.float(), A, dt)), "one of two": (lambda *t: lm_engine_amd.delta_rule_gates(*t)[0], (a, b, A, dt)),
    }  # fmt: skip
    o, z, nw = r(2, 70, 2, 64), r(2, 70, 128), r(64)
    norm = lambda o, z, w=None: lm_engine_amd.gated_rmsnorm(o, z, w, 1e-5)  # noqa: E731
    yield "norm_bwd", {
        "plain": (norm, (o, z, nw)), "no weight": (norm, (o, z)), "no gate": (lambda o, w: norm(o, None, w), (o, nw)), "gate by heads": (norm, (o, z.view(2, 70, 2, 64), nw)),
        "gate slice": (norm, (o, r(2, 70, 140)[..., 4:132], nw)), "gate slice off its boundary": (norm, (o, r(2, 70, 140)[..., 3:131], nw)), "o strided": (norm, (r(2, 2, 70, 64).transpose(1, 2), z, nw)),
        "fp32": (norm, (o.float(), z.float(), nw.float())), "fp32 weight": (norm, (o, z, nw.float())),
    }  # fmt: skip
    for T in (128, 130):
        unit = lambda x: torch.nn.functional.normalize(x, dim=-1)  # noqa: E731
        q, k, v = unit(r(2, T, 2, 64)), unit(r(2, T, 2, 64)), r(2, T, 2, 64)
        g, beta, h = -torch.rand(2, T, 2, generator=gen).cuda(), torch.rand(2, T, 2, generator=gen).to(BF16).cuda(), torch.randn(2, 2, 64, 64, generator=gen).cuda()
        qkv = 0.1 * r(2, T, 3 * 128)
        blocks = [x.view(2, T, 2, 64) for x in qkv.split(128, dim=-1)]

        def op(**kw):
            def run(q, k, v, g=None, beta=None, h=None):
                o, ht = lm_engine_amd.chunk_gated_delta_rule(q, k, v, g, beta, initial_state=h, **kw)
                return o if ht is None else torch.cat([o.flatten().float(), ht.flatten()])

            return run

        cu = lambda *ends: torch.tensor(ends, dtype=torch.int32).cuda()  # noqa: E731
        one = tuple(t[:1] for t in (q, k, v, g, beta))
        yield "delta_rule_bwd", {
            "plain": (op(use_qk_l2norm_in_kernel=True), (q, k, v, g, beta)), "no l2norm": (op(), (q, k, v, g, beta)), "ungated": (op(), (q, k, v)), "beta fp32": (op(), (q, k, v, g, beta.float())),
            "states": (op(output_final_state=True, use_qk_l2norm_in_kernel=True), (q, k, v, g, beta, h)), "scale": (op(scale=0.3), (q, k, v, g, beta)), "blocks of one tensor": (op(), (*blocks, g, beta)), "blocks, shared heads": (op(), (blocks[0][:, :, :1], blocks[1][:, :, :1], blocks[2], g, beta)),
            "strided q": (op(), (unit(r(2, 2, T, 64)).transpose(1, 2), k, v, g, beta)), "shared heads": (op(use_qk_l2norm_in_kernel=True), (q[:, :, :1], k[:, :, :1], v, g, beta)),
            "packed": (op(cu_seqlens=cu(0, 3, T), output_final_state=True), (*one, h)), "packed, empty ones": (op(cu_seqlens=cu(0, 0, 70, 70, T)), one), "packed, tokens left over": (op(cu_seqlens=cu(0, 70, T - 9)), one),
            "packed, int64 prefix": (op(cu_seqlens=cu(0, 3, T).long()), one), "padded": (op(cu_seqlens=cu(0, 70, 70 + T), left_padded=True), (q, k, v, g, beta)), "fp32": (op(), tuple(t.float() for t in (q, k, v, g, beta))),
            "V = 96": (op(), (q, k, r(2, T, 2, 96), g, beta)),
        }  # fmt: skip


# Which of the three gradients below the native path takes: not one value for all elements, in no case, nor rows that the norm
# would have to copy, nor operands that need a conversion.  (): the Python code does not ask.
_BACKWARD_TAKES = {"conv_bwd": (True, True, False), "gates_bwd": (True, True, False), "norm_bwd": (True, False, False), "delta_rule_bwd": (True, True, False)}
_BACKWARD_TAKES_OF_FORM = {
    ("conv_bwd", "state"): (), ("gates_bwd", "bf16 decay"): (False, False, False), ("gates_bwd", "one of two"): (True, False, False),
    ("norm_bwd", "o strided"): (False, False, False), ("norm_bwd", "gate slice off its boundary"): (False, False, False),
    ("delta_rule_bwd", "packed, int64 prefix"): (False, False, False), ("delta_rule_bwd", "fp32"): (), ("delta_rule_bwd", "V = 96"): (),
}  # fmt: skip


def test_backward_passes_end_as_they_do_without_the_native_path(monkeypatch):
    """The gradients of every form are the same bits with the native host path and without it, for a gradient that lies as
    the output does, a column block of a wider one, and one value for all elements; and every form takes the path it is meant to."""
    from lm_engine_amd import backward, conv, layer_ops, ops

    differ = []
    for name, forms in _training_forms():
        for form, (function, operands) in forms.items():
            outcomes = []
            print(f"case: {name}, {form}", flush=True)
            for on in (True, False):
                path = _NativePath(on)
                with monkeypatch.context() as m:
                    for module in (backward, conv, layer_ops, ops):
                        m.setattr(module, "host", lambda path=path: path)
                    leaves = [x.detach().requires_grad_(True) for x in operands]
                    out = function(*leaves)
                    path.took.clear()
                    wide = torch.randn(*out.shape[:-1], 2 * out.size(-1) + 8, generator=torch.Generator().manual_seed(4)).to(out.dtype).cuda()
                    results = []
                    for d in (wide[..., : out.size(-1)].contiguous(), wide[..., 8 : 8 + out.size(-1)], torch.ones((), dtype=out.dtype).cuda().expand(out.shape)):
                        results += [x.clone() for x in torch.autograd.grad(out, leaves, d, retain_graph=True, allow_unused=True) if x is not None]
                outcomes.append(results)
                takes = _BACKWARD_TAKES_OF_FORM.get((name, form), _BACKWARD_TAKES[name])
                assert path.took == [on and x for x in takes], f"{name}, {form}: the path under test was not the one taken: {path.took}"
            if not all(x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y) for x, y in zip(*outcomes)) or len(outcomes[0]) != len(outcomes[1]):
                differ.append((name, form))
    torch.cuda.synchronize()
    assert not differ, differ


@pytest.mark.parametrize("S, dtype", [(2, BF16), (70, BF16), (130, torch.float32), (1100, BF16)])
@pytest.mark.parametrize("B", [1, 3])
def test_the_layers_front_in_one_launch_gives_the_bits_of_its_steps(B, S, dtype, monkeypatch):
    """Convolution, gates and the mask's prefix sums: short walks over the tokens, integer masks of every type and layout, a single
    row (whose mask the convolution does not apply), rows without a token, and what is refused."""
    from lm_engine_amd import layer

    x = _layer_operands(B, S)
    x = {n: t.to(dtype) if isinstance(t, torch.Tensor) and t.dtype == BF16 else t for n, t in x.items()}
    wide = torch.randn(B, S, 2 + 2 + 128, generator=torch.Generator().manual_seed(5)).to(dtype).cuda()
    state = torch.randn(B, 384, 3, generator=torch.Generator().manual_seed(6)).to(dtype).cuda()
    lengths = torch.tensor([S, 0, S // 2][:B])
    mask = (torch.arange(S)[None] >= S - lengths[:, None]).cuda()
    forms = {
        "no mask": {}, "cache": dict(cache=(None, None)), "carried": dict(cache=(state, None)), "slices": dict(a=wide[..., :2], b=wide[..., 2:4], gate=wide[..., 4:]),
        "int64": dict(attention_mask=mask.long()), "int32": dict(attention_mask=mask.int()), "uint8": dict(attention_mask=mask.byte()), "bool": dict(attention_mask=mask),
        "transposed mask": dict(attention_mask=mask.long().t().contiguous().t(), cache=(None, None)), "expanded mask": dict(attention_mask=torch.ones(B, 1, dtype=torch.int32).cuda().expand(B, S)),
        "mask in fp32": dict(attention_mask=mask.float()), "mask of another shape": dict(attention_mask=mask[:, 1:].long()), "a of fewer tokens": dict(a=x["a"][:, 1:], b=x["b"][:, 1:]),
        "2-D weight": dict(conv_weight=x["conv_weight"][:, 0]), "3 taps": dict(conv_weight=x["conv_weight"][..., 1:].contiguous()), "no activation": dict(conv_activation=None), "negative eigenvalues": dict(allow_neg_eigval=True),
    }  # fmt: skip
    for form, over in forms.items():
        print(f"case: layer's front, {B} x {S}, {form}", flush=True)
        outcomes = []
        for on in (True, False):
            took = []

            class Path:
                def __getattr__(self, name):
                    return getattr(_host.host(), name)

                def layer_front(self, *args, on=on, took=took):
                    result = _host.host().layer_front(*args) if on else None
                    took.append(result is not None)
                    return result

            with monkeypatch.context() as m:
                m.setattr(layer, "host", Path)
                outcomes.append(_outcome(lambda: lm_engine_amd.gated_deltanet_mixing(**{**x, **over})))
            assert form == "a of fewer tokens" or took == [on and form not in ("mask in fp32", "mask of another shape")]
        (one, steps), refused = outcomes, isinstance(outcomes[0], tuple)
        assert refused == isinstance(steps, tuple) and len(one) == len(steps)
        assert one == steps if refused else all((p is None and q is None) or torch.equal(p, q) for p, q in zip(one, steps)), form
    torch.cuda.synchronize()


@pytest.mark.parametrize(
    "B, S, HK, H, K, V, mask_dtype",
    # many short rows: the gates on one plane of workgroups and on several; rows of a mask four to a wave, whole and cut, parts of rows
    [(1024, 3, 4, 4, 64, 64, None), (300, 17, 2, 4, 64, 64, None), (64, 5, 4, 4, 64, 64, torch.int64), (64, 130, 4, 4, 64, 64, torch.bool), (17, 65, 2, 2, 64, 64, torch.int32),
     (16, 1, 2, 2, 64, 64, torch.int64), (5, 300, 2, 2, 64, 64, torch.uint8), (2, 1000, 2, 2, 64, 64, torch.int64),
     # walks of 8 tokens that end within one, over several groups of channels, the last one whole and cut
     (3, 4797, 5, 5, 64, 64, None), (3, 3201, 6, 6, 64, 128, None), (3, 4797, 5, 5, 64, 64, torch.int64), (3, 4797, 5, 5, 64, 64, torch.int32), (3, 4797, 5, 5, 64, 64, torch.bool), (3, 3201, 6, 6, 64, 128, torch.int64)],
)  # fmt: skip
def test_the_layers_front_of_many_rows_and_of_long_walks(B, S, HK, H, K, V, mask_dtype):
    from lm_engine_amd.layer_ops import padding_mask

    gen = torch.Generator("cuda").manual_seed(B + S)
    r = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(BF16)  # noqa: E731
    C = 2 * HK * K + H * V
    x, ab, w, bias, A, dt = r(B, S, C), r(B, S, 2 * H + 3), 0.3 * r(C, 1, 4), 0.1 * r(C), r(H).float(), r(H).float()
    state, a, b, mask, stream, native = r(B, C, 3), ab[..., :H], ab[..., H : 2 * H], None, _host.raw_stream(0), _host.host()
    if mask_dtype is not None:
        lengths = torch.randint(0, S + 1, (B,), generator=torch.Generator().manual_seed(S))
        mask = (torch.arange(S) >= S - lengths[:, None]).to(mask_dtype).cuda()
    print(f"case: layer's front, {B} x {S} tokens, {C} channels, mask {mask_dtype}", flush=True)
    *front, prefix = native.layer_front(stream, x, w, bias, state, mask, True, 1, a, b, A, dt, 1.0)
    bits, wanted = (None, None) if mask is None else padding_mask(mask, BF16)
    steps = [*native.conv(stream, x, w, bias, state, bits, True, 1), *native.gates(stream, a, b, A, dt, 1.0)]
    assert all(torch.equal(p, q) for p, q in zip(front, steps)) and (mask is None) == (prefix is None)
    assert mask is None or torch.equal(prefix, wanted) and torch.equal(wanted.cpu(), torch.nn.functional.pad(lengths.cumsum(0), (1, 0)).int())
