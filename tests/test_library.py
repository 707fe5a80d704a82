"""Host-side checks that need no GPU: the C-ABI library loads, exports what include/gdn_hip.h
declares, agrees with the ctypes mirror of the argument struct, and rejects bad arguments
before anything is launched."""

import ctypes
import hashlib
import os
import re
import subprocess
import sys
import tempfile
import threading
import time

import pytest
import torch

import lm_engine_amd
from lm_engine_amd import _lib
from lm_engine_amd.kernels import Kernel, enable_kernels, is_kernel_allowed


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gdn_hip.h")


def _declared_functions() -> list[str]:
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.findall(r"\b(gdn_[a-z0-9_]+)\s*\(", text)


def test_library_exports_every_declared_symbol():
    lib = _lib.load_library()
    declared = set(_declared_functions())
    assert declared == set(_lib.EXPORTED_SYMBOLS), declared
    for name in declared:
        assert hasattr(lib, name), name
    assert lib.gdn_abi_version() == _lib.GDN_ABI_VERSION


def test_struct_layout_matches_the_header():
    source = r"""
    #include <stdio.h>
    #include <stddef.h>
    #include "gdn_hip.h"
    int main(void) {
        printf("%zu %zu %zu %zu %zu %zu %zu\n", sizeof(gdn_args), offsetof(gdn_args, workspace_bytes),
               offsetof(gdn_args, q_stride_b), offsetof(gdn_args, o_stride_h), offsetof(gdn_args, B),
               offsetof(gdn_args, flags), offsetof(gdn_args, scale));
        printf("%zu %zu\n", offsetof(gdn_args, spin_limit), offsetof(gdn_args, error_word));
        printf("%zu %zu %zu %zu %zu\n", sizeof(gdn_conv_args), offsetof(gdn_conv_args, final_state),
               offsetof(gdn_conv_args, x_stride_b), offsetof(gdn_conv_args, B), offsetof(gdn_conv_args, activation));
        return 0;
    }
    """
    with tempfile.TemporaryDirectory() as tmp:
        src, exe = os.path.join(tmp, "layout.c"), os.path.join(tmp, "layout")
        open(src, "w").write(source)
        subprocess.run(["gcc", f"-I{os.path.dirname(HEADER)}", src, "-o", exe], check=True)
        values = [int(x) for x in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()]
    A = _lib.GdnArgs
    Cv = _lib.GdnConvArgs
    assert values == [ctypes.sizeof(A), A.workspace_bytes.offset, A.q_stride_b.offset, A.o_stride_h.offset,
                      A.B.offset, A.flags.offset, A.scale.offset, A.spin_limit.offset, A.error_word.offset,
                      ctypes.sizeof(Cv), Cv.final_state.offset, Cv.x_stride_b.offset, Cv.B.offset,
                      Cv.activation.offset]  # fmt: skip


# sha256 (16 digits) of the header's structs without comments, by the version that they had
STRUCTS_OF_VERSION = {2: "7652088ae5119dd4", 3: "19be2afcc6940cb1"}


def test_a_change_of_the_structs_comes_with_a_new_version():
    """A caller built against an older header is told so by the version: also where a reserved field became one that is read
    (callers were not asked to clear it)."""
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    structs = re.findall(r"typedef struct \w+ \{.*?\} \w+;", text, flags=re.S)
    digest = hashlib.sha256(" ".join(" ".join(structs).split()).encode()).hexdigest()[:16]
    version = int(re.search(r"#define GDN_ABI_VERSION (\d+)", text).group(1))
    assert STRUCTS_OF_VERSION.get(version) == digest, f"version {version}: structs {digest}"


def test_layer_ops_reject_bad_arguments_before_any_launch():
    lib = _lib.load_library()
    g = _lib.GdnGateArgs()
    g.a = g.b = g.A_log = g.dt_bias = g.g = g.beta = 0x1000
    g.tokens, g.H, g.a_stride, g.b_stride, g.dtype, g.beta_scale = 4, 8, 8, 8, _lib.GDN_BF16, 1.0
    for over, status in [(dict(a=None), -1), (dict(tokens=0), -2), (dict(a_stride=4), -2), (dict(dtype=5), -3)]:
        a = _lib.GdnGateArgs.from_buffer_copy(g)
        for name, value in over.items():
            setattr(a, name, value)
        assert lib.gdn_gates_fwd(ctypes.byref(a), None) == status, over
    n = _lib.GdnNormArgs()
    n.o, n.y = 0x1000, 0x2000
    n.tokens, n.H, n.V, n.dtype, n.w_dtype, n.eps = 4, 2, 64, _lib.GDN_BF16, _lib.GDN_F32, 1e-6
    n.o_stride_t = n.y_stride_t = 128
    for over, status in [(dict(o=None), -1), (dict(V=0), -2), (dict(V=20), -3), (dict(V=1024), -3), (dict(o_stride_t=64), -2),
                         (dict(o=0x1002), -4), (dict(gate=0x3008, gate_stride_t=128), -4), (dict(o_stride_t=132), -4)]:  # fmt: skip
        a = _lib.GdnNormArgs.from_buffer_copy(n)
        for name, value in over.items():
            setattr(a, name, value)
        assert lib.gdn_gated_rmsnorm_fwd(ctypes.byref(a), None) == status, over


def test_flags_of_the_chunk_local_gradients_are_checked_before_any_launch():
    lib = _lib.load_library()
    flags = {name: int(value, 0) for name, value in re.findall(r"#define GDN_LOCAL_(\w+) (0x\w+)", open(HEADER).read())}
    assert flags == {"DBETA_BF16": 0x100, "RAGGED_ROWS": 0x200}
    ragged = flags["RAGGED_ROWS"]

    def status(flag, **over):
        a = _lib.GdnChunkLocalArgs()
        for name, kind in a._fields_:
            if kind is ctypes.c_void_p and name not in ("seq_start", "seq_len", "rk"):
                setattr(a, name, 0x1000)  # never dereferenced: rq without rk is refused, behind the flags
        a.saves_dtype, a.dstates_dtype, a.saves_sliced = _lib.GDN_BF16 | flag, _lib.GDN_BF16, 1
        a.chunks, a.K, a.V, a.H, a.NC, a.scale = 6, 64, 64, 1, 3, 1.0
        for name, value in over.items():
            setattr(a, name, value)
        return lib.gdn_chunk_bwd_local(ctypes.byref(a), None)

    assert status(0x400) == status(ragged | 0x800) == -3
    for T_rows in (0, 1, 64, 128, 193, -5):
        assert status(ragged, T_rows=T_rows) == -2, T_rows
    assert status(ragged, T_rows=150, seq_start=0x1000, seq_len=0x1000) == -2
    for flag, T_rows in ((0, 0), (0, 150), (flags["DBETA_BF16"], -5), (ragged, 129), (ragged, 192), (ragged | 0x20000, 150)):
        assert status(flag, T_rows=T_rows, H=2) == -1, (flag, T_rows)


def test_convolution_rejects_bad_arguments_before_any_launch():
    lib = _lib.load_library()

    def conv_args(**over):
        a = _lib.GdnConvArgs()
        a.x, a.y, a.weight = 0x1000, 0x2000, 0x3000  # never dereferenced
        a.B, a.S, a.C, a.kernel_size = 2, 8, 16, 4
        a.x_stride_s = a.y_stride_s = 16
        a.x_stride_b = a.y_stride_b = 128
        a.dtype, a.w_dtype, a.activation = _lib.GDN_BF16, _lib.GDN_BF16, _lib.GDN_ACT_SILU
        for name, value in over.items():
            setattr(a, name, value)
        return a

    for over, status in [
        (dict(x=None), -1),
        (dict(S=0), -2),
        (dict(kernel_size=5), -3),
        (dict(kernel_size=1), -3),
        (dict(C=12), -3),
        (dict(activation=7), -3),
        (dict(x_stride_s=20), -4),
        (dict(x=0x1008), -4),
        (dict(y=0x1000), -2),
        (dict(x_stride_s=8), -2),
        (dict(S=65535 * 64), -3),
        # more threads than a grid holds, in walks of 8 tokens (bf16) and of 4 (fp32)
        (dict(S=65535 * 64 - 1, C=1 << 17, x_stride_s=1 << 17, y_stride_s=1 << 17), -3),
        (dict(S=65535 * 64 - 1, C=1 << 15, x_stride_s=1 << 15, y_stride_s=1 << 15, dtype=_lib.GDN_F32, w_dtype=_lib.GDN_F32), -3),
    ]:
        assert lib.gdn_causal_conv1d_fwd(ctypes.byref(conv_args(**over)), None) == status, over


def _args(**over):
    a = _lib.GdnArgs()
    fake = 0x1000  # never dereferenced: validation fails before any launch
    a.q = a.k = a.v = a.o = fake
    a.B, a.T, a.H, a.K, a.V, a.N = 1, 8, 2, 64, 64, 1
    a.q_stride_h = a.k_stride_h = 64
    a.v_stride_h = a.o_stride_h = 64
    a.q_stride_t = a.k_stride_t = a.v_stride_t = a.o_stride_t = 128
    a.q_stride_b = a.k_stride_b = a.v_stride_b = a.o_stride_b = 1024
    a.dtype, a.beta_dtype, a.scale = _lib.GDN_BF16, _lib.GDN_BF16, 0.125
    for name, value in over.items():
        setattr(a, name, value)
    return a


@pytest.mark.parametrize(
    "over, status",
    [
        (dict(q=None), -1),
        (dict(T=0), -2),
        (dict(N=3), -2),
        (dict(K=48), -3),
        (dict(V=40), -3),
        (dict(dtype=7), -3),
        (dict(q_stride_t=129), -4),
        (dict(v=0x1004), -4),
        (dict(cu_seqlens=0x2000, B=2, N=2), -6),
        (dict(flags=_lib.GDN_FLAG_LEFT_PADDED), -1),  # left-padded needs the prefix sums
        (dict(flags=_lib.GDN_FLAG_LEFT_PADDED, cu_seqlens=0x2000, B=2, N=3), -2),  # one sequence per row
        (dict(q_stride_h=32), -2),
    ],
)
def test_bad_arguments_are_rejected_before_launch(over, status):
    lib = _lib.load_library()
    a = _args(**over)
    assert lib.gdn_recurrent_fwd(ctypes.byref(a), None) == status
    assert lib.gdn_chunk_fwd(ctypes.byref(a), None) == status
    assert _lib.strerror(status) != "unknown gdn status"


STEP, TOKENS = 1, 2


@pytest.mark.parametrize(
    "over, kernels",
    [
        # fixed-length batches and rows of a left-padded one: T tokens each
        (dict(T=1), STEP), (dict(T=2), TOKENS), (dict(T=11, B=256, N=256, H=32, V=128), STEP), (dict(T=12, B=256, N=256, H=32, V=128), TOKENS),
        (dict(T=40, B=40, N=40, cu_seqlens=0x2000, flags=_lib.GDN_FLAG_LEFT_PADDED), TOKENS),
        # packed: T is the tokens of all sequences
        (dict(T=256, N=256, cu_seqlens=0x2000), STEP), (dict(T=12, N=12, cu_seqlens=0x2000), STEP), (dict(T=12, N=20, cu_seqlens=0x2000), STEP),
        (dict(T=257, N=256, H=32, K=128, V=128, cu_seqlens=0x2000), STEP | TOKENS),
        (dict(T=256 * 48 - 1, N=256, H=32, K=128, V=128, cu_seqlens=0x2000), STEP | TOKENS),
        (dict(T=256 * 48, N=256, H=32, K=128, V=128, cu_seqlens=0x2000), TOKENS),
        (dict(T=12, N=4, H=16, K=128, V=128, cu_seqlens=0x2000), TOKENS),  # few states
        (dict(T=5000, N=4, H=16, K=128, V=128, cu_seqlens=0x2000), TOKENS),
    ],
)  # fmt: skip
def test_kernels_of_the_recurrent_forward_by_tokens_per_sequence(over, kernels):
    assert _lib.load_library().gdn_recurrent_fwd_kernels(ctypes.byref(_args(**over))) == kernels


def test_chunk_fwd_needs_a_workspace():
    lib = _lib.load_library()
    a = _args(T=128, K=128, V=128, q_stride_h=128, k_stride_h=128, v_stride_h=128, o_stride_h=128,
              q_stride_t=256, k_stride_t=256, v_stride_t=256, o_stride_t=256, q_stride_b=256 * 128,
              k_stride_b=256 * 128, v_stride_b=256 * 128, o_stride_b=256 * 128)  # fmt: skip
    need = lib.gdn_workspace_bytes(ctypes.byref(a))
    assert need > 0
    assert lib.gdn_chunk_fwd(ctypes.byref(a), None) == -5
    a.workspace, a.workspace_bytes = 0x10000, need - 1
    assert lib.gdn_chunk_fwd(ctypes.byref(a), None) == -5
    a.dtype = _lib.GDN_F32  # fp32 inputs have no chunk kernel
    assert lib.gdn_workspace_bytes(ctypes.byref(a)) == 0
    assert lib.gdn_chunk_fwd(ctypes.byref(a), None) == -3


def test_python_wrapper_validates_and_never_falls_back():
    q = torch.zeros(1, 8, 2, 64, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="GPU only"):
        lm_engine_amd.fused_recurrent_gated_delta_rule(q=q, k=q, v=q)
    with pytest.raises(ValueError, match="shape of q"):
        lm_engine_amd.chunk_gated_delta_rule(q=q, k=q[:, :4], v=q)
    with pytest.raises(ValueError, match="head_first"):
        lm_engine_amd.chunk_gated_delta_rule(q=q, k=q, v=q, head_first=True)


def test_missing_library_fails_loudly(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIBRARY_PATH", "/nonexistent/libgdn_hip.so")
    with pytest.raises(_lib.GdnLibraryError, match="no fallback"):
        _lib.load_library()


def test_package_imports_on_a_torch_build_without_gpu_support():
    code = ("import torch; del torch._C._cuda_getCurrentRawStream\n"
            "import lm_engine_amd, oracle; x = torch.zeros(1, 8, 2, 64, dtype=torch.bfloat16)\n"
            "try: lm_engine_amd.chunk_gated_delta_rule(x, x, x)\n"
            "except ValueError as e: print(e)")  # fmt: skip
    run = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert run.returncode == 0 and "GPU only" in run.stdout, run.stderr


def test_warmup_of_the_benchmark_is_not_spent_on_loading(monkeypatch):
    """The first call of a process loads libraries and code objects for longer than the warm-up lasts: it comes before the clock."""
    import bench

    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    made = []
    bench.device_warmup(lambda: time.sleep(0.002 if made else 0.2) or made.append(1), ms=40.0)
    assert len(made) >= 12


def test_threads_that_ask_first_share_one_error_word(monkeypatch):
    """The look at a device's error word goes to the address of the word that the library is given, also when several threads
    make their first call at once (the slow allocation lets both in; no device is touched)."""
    from lm_engine_amd import ops

    zeros = torch.zeros

    def slow_zeros(*args, **kwargs):
        word = zeros(*args, **kwargs)
        time.sleep(0.05 * (1 + len(made)))
        made.append(word)
        return word

    made, got = [], []
    monkeypatch.setattr(ops, "_ERROR_WORDS", {})
    monkeypatch.setattr(ops, "_ERROR_PEEKS", {})
    monkeypatch.setattr(torch, "zeros", slow_zeros)
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    threads = [threading.Thread(target=lambda: got.append(ops._error_word(torch.device("cuda", 3)))) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == 3 and all(word is ops._ERROR_WORDS[3] for word in got)
    assert ctypes.addressof(ops._ERROR_PEEKS[3]) == ops._ERROR_WORDS[3].data_ptr()


def test_kernel_flag_registry_follows_the_reference_convention():
    assert is_kernel_allowed(Kernel.gated_delta_rule)
    with enable_kernels([], reset=True):
        assert not is_kernel_allowed(Kernel.gated_delta_rule)
        q = torch.zeros(1, 8, 2, 64, dtype=torch.bfloat16)
        with pytest.raises(RuntimeError, match="no other implementation"):
            lm_engine_amd.fused_recurrent_gated_delta_rule(q=q, k=q, v=q)
        with enable_kernels([Kernel.gated_delta_rule]):
            assert is_kernel_allowed(Kernel.gated_delta_rule)
        assert not is_kernel_allowed(Kernel.gated_delta_rule)
    assert is_kernel_allowed(Kernel.gated_delta_rule)


def test_a_backward_under_a_switched_off_kernel_is_refused(monkeypatch):
    """Of the operator, the gates and the gated norm: ahead of anything that the native host path would launch."""
    from lm_engine_amd import backward, layer_ops

    class NotAsked:
        def __getattr__(self, name):
            raise AssertionError(f"{name} was called")

    for module in (backward, layer_ops):
        monkeypatch.setattr(module, "host", NotAsked)
    x, h = torch.zeros(1, 64, 2, 64, dtype=torch.bfloat16), torch.zeros(2)
    a = x[..., 0]
    rule = lambda: backward._backward_on_kernels(x, x, x, None, None, x, None, 1.0, None, False, None, False, False)  # noqa: E731
    with enable_kernels([], reset=True):
        for call in (rule, lambda: layer_ops._delta_rule_gates_backward(a, a, h, h, a, a, False),
                     lambda: layer_ops._gated_rmsnorm_backward(x, None, None, None, x)):  # fmt: skip
            with pytest.raises(RuntimeError, match="no other implementation"):
                call()


def test_fused_launch_flag_is_on_by_default_and_can_be_switched_off():
    fused = Kernel.gated_delta_rule_fused_launch
    assert is_kernel_allowed(fused)
    with enable_kernels([Kernel.gated_delta_rule], reset=True):
        assert not is_kernel_allowed(fused) and is_kernel_allowed(Kernel.gated_delta_rule)
    assert is_kernel_allowed(fused)
    assert _lib.GDN_FLAG_FUSED_LAUNCH == 8 and _lib.GDN_FLAG_READY_FLAGS_CLEAR == 16


def test_kernel_flag_env_variable():
    code = "from lm_engine_amd.kernels import Kernel, is_kernel_allowed; print(is_kernel_allowed(Kernel.gated_delta_rule))"
    run = lambda env: subprocess.run([sys.executable, "-c", code], env={**os.environ, **env}, cwd=ROOT,
                                     capture_output=True, text=True, check=True).stdout.strip()  # noqa: E731  # fmt: skip
    assert run({"ENABLE_KERNELS": "rmsnorm"}) == "False"
    assert run({"ENABLE_KERNELS": "rmsnorm, gated_delta_rule"}) == "True"
    assert run({"ENABLE_ALL_KERNELS": "1"}) == "True"


def test_fla_shim_resolves_the_reference_imports():
    from lm_engine_amd import install_as_fla, uninstall_fla_shim

    install_as_fla()
    try:
        from fla.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule
        import fla  # noqa: F401  (the reference's availability probe, lm_engine/utils/packages.py:56-61)

        assert chunk_gated_delta_rule is lm_engine_amd.chunk_gated_delta_rule
        assert fused_recurrent_gated_delta_rule is lm_engine_amd.fused_recurrent_gated_delta_rule
    finally:
        uninstall_fla_shim()
    assert "fla" not in sys.modules


def test_noalloc_entry_point_rejects_shapes_beyond_its_scratch():
    lib = _lib.load_library()
    args = _lib.GdnArgs()
    args.q = args.k = args.v = args.o = 0x1000
    args.B, args.T, args.H, args.K, args.V, args.N = 8, 8192, 16, 128, 128, 8
    args.chunk, args.dtype, args.beta_dtype, args.scale = 64, _lib.GDN_BF16, _lib.GDN_BF16, 1.0
    for name in ("q", "k", "v", "o"):
        setattr(args, f"{name}_stride_b", 8192 * 16 * 128)
        setattr(args, f"{name}_stride_t", 16 * 128)
        setattr(args, f"{name}_stride_h", 128)
    assert lib.gdn_workspace_bytes(ctypes.byref(args)) > _lib.GDN_NOALLOC_SCRATCH_BYTES
    assert lib.gdn_chunk_fwd_noalloc(ctypes.byref(args), None) == -5  # GDN_ERR_WORKSPACE, before any launch


def test_opaque_operators_are_registered_with_shape_only_implementations():
    # what torch.compile captures in place of the ctypes launches: one torch.library operator per kernel, each with a
    # fake implementation (run here on meta tensors: no kernel is launched)
    import torch

    from lm_engine_amd import _opaque  # noqa: F401

    ops = torch.ops.lm_engine_amd
    for name in ("gated_delta_rule_forward", "gated_delta_rule_backward", "gated_delta_rule_decode_",
                 "causal_conv1d_forward", "causal_conv1d_backward", "delta_rule_gates_forward",
                 "delta_rule_gates_backward", "gated_rmsnorm_forward", "gated_rmsnorm_backward"):  # fmt: skip
        assert hasattr(ops, name), name
    meta = lambda *shape, dtype=torch.bfloat16: torch.empty(*shape, dtype=dtype, device="meta")  # noqa: E731
    B, T, H, K, V = 2, 130, 3, 128, 64
    q, k, v = meta(B, T, H, K), meta(B, T, H, K), meta(B, T, H, V)
    g, beta, h0 = meta(B, T, H, dtype=torch.float32), meta(B, T, H), meta(B, H, K, V, dtype=torch.float32)
    o, ht = ops.gated_delta_rule_forward(q, k, v, g, beta, h0, None, "chunk", None, True, False, False)
    assert tuple(o.shape) == (B, T, H, V) and o.dtype == torch.bfloat16
    assert tuple(ht.shape) == (B, H, K, V) and ht.dtype == torch.float32
    o, ht = ops.gated_delta_rule_forward(q, k, v, None, None, None, None, "chunk", 0.5, False, True, False)
    assert ht.numel() == 0
    cu = torch.empty(4, dtype=torch.int32, device="meta")
    _, ht = ops.gated_delta_rule_forward(q[:1], k[:1], v[:1], None, None, None, cu, "chunk", None, True, False, False)
    assert tuple(ht.shape) == (3, H, K, V)
    grads = ops.gated_delta_rule_backward(q, k, v, g, None, h0, None, o, None, None, False, False)
    assert [tuple(x.shape) for x in grads] == [(B, T, H, K), (B, T, H, K), (B, T, H, V), (B, T, H), (0,), (B, H, K, V)]
    y, state = ops.causal_conv1d_forward(meta(B, T, 96), meta(96, 4), None, None, None, True, "silu")
    assert tuple(y.shape) == (B, T, 96) and tuple(state.shape) == (B, 96, 3)
    gg, bb = ops.delta_rule_gates_forward(meta(B, T, H), meta(B, T, H), meta(H, dtype=torch.float32),
                                          meta(H, dtype=torch.float32), False)  # fmt: skip
    assert gg.dtype == torch.float32 and bb.dtype == torch.bfloat16 and tuple(gg.shape) == (B, T, H)
    assert tuple(ops.gated_rmsnorm_forward(meta(B, T, H, V), meta(B, T, H * V), meta(V), None).shape) == (B, T, H, V)


def test_padding_masks_of_many_rows_do_not_go_through_one_workgroup():
    """Up to 64 rows and 64 K elements the one launch is the faster way at every size; 1024 rows took it 3.5 times as long as torch."""
    from lm_engine_amd.layer_ops import _one_launch_mask

    for B, S, one in [(1, 1, True), (64, 1024, True), (65, 1, False), (256, 256, False), (1024, 8, False), (64, 1025, False), (1, 1 << 16, True)]:
        for dtype in (torch.int64, torch.int32, torch.uint8, torch.bool):
            assert _one_launch_mask(B, S, dtype, torch.bfloat16) == one, (B, S)
    assert not _one_launch_mask(2, 8, torch.float32, torch.bfloat16) and not _one_launch_mask(2, 8, torch.int64, torch.float16)
    assert not _one_launch_mask(0, 8, torch.int64, torch.bfloat16) and not _one_launch_mask(2, 0, torch.int64, torch.bfloat16)
