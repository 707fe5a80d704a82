"""The native host path of the inference entry points (csrc/gdn_host.cpp): what it hands on to the Python code, what it raises,
and what it leaves behind.  The library's entry points are replaced by small stand-ins where a test needs a status or a look
at the thread's state: nothing is launched then."""

import contextlib
import ctypes
import sys

import pytest
import torch

import lm_engine_amd
from lm_engine_amd import _host, _lib


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
