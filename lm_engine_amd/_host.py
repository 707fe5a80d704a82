"""Loads ``gdn_host.so``, the host path of the entry points and their backward passes (csrc/gdn_host.cpp), and hands it the addresses of the
HIP library's entry points, so that both sides work on the one loaded copy.

Its functions take the operands of a call and return its results, or None where the Python code has to convert,
differentiate or report.  Like the HIP library it is built by ``python -m lm_engine_amd.build``, and a GPU call without it
fails loudly."""

from __future__ import annotations

import ctypes
import importlib
import os

import torch

from . import _lib


MODULE_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gdn_host.so")

_BOUND = ("gdn_layer_step", "gdn_layer_step_tiles", "gdn_causal_conv1d_fwd", "gdn_gates_fwd", "gdn_gated_rmsnorm_fwd",
          "gdn_recurrent_fwd", "gdn_chunk_fwd", "gdn_workspace_bytes", "gdn_chunk_fwd_is_one_launch", "gdn_chunk_bwd_sweeps",
          "gdn_chunk_bwd_sweeps_workspace_bytes", "gdn_chunk_bwd_local", "gdn_causal_conv1d_bwd", "gdn_gates_bwd",
          "gdn_gated_rmsnorm_bwd", "gdn_column_sums", "gdn_fold_heads", "gdn_layer_front")  # fmt: skip

# device index -> hipStream_t of the calling thread's current stream (a torch build without GPU support has no such function,
# nor a device tensor that would lead here)
raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)

_module = None


def host():
    global _module
    if _module is None:
        lib = _lib.load_library()
        if not os.path.exists(MODULE_PATH):
            raise _lib.GdnLibraryError(f"{MODULE_PATH} is missing: run `python -m lm_engine_amd.build`")
        module = importlib.import_module(".gdn_host", __package__)
        module.bind(_lib.check_status, *(ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _BOUND))
        _module = module
    return _module
