"""The library's own rules of dispatch, called as they are (host code, no GPU): which kernel a launch of these sizes takes."""

from __future__ import annotations

import ctypes

from lm_engine_amd import _lib


class ScanPlan(ctypes.Structure):  # gdn_chunk_common.h
    _fields_ = [("nw", ctypes.c_int), ("half", ctypes.c_bool), ("split_keys", ctypes.c_bool), ("direct", ctypes.c_bool), ("staged_saves", ctypes.c_bool), ("no_output", ctypes.c_bool)]


class SaveRequest(ctypes.Structure):
    _fields_ = [(name, ctypes.c_bool) for name in ("no_output", "has_state", "has_vnew", "state_bf16", "vnew_bf16")] + [("save_every", ctypes.c_int)]


def scan_plan(K, chains, T, V, packed=False, cus=256) -> ScanPlan:
    """Of a forward that saves nothing."""
    rule = _lib.load_library()["_ZN3gdn9plan_scanEiliibbiiRKNS_11SaveRequestE"]
    rule.restype, rule.argtypes = ScanPlan, [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_bool, ctypes.c_bool, ctypes.c_int, ctypes.c_int, ctypes.POINTER(SaveRequest)]
    return rule(K, chains, T, V, packed, False, 0, cus, ctypes.byref(SaveRequest(False, True, True, False, False, 1)))


def sweep_columns(N, H, V, longest, chunks, packed=False, padded=False, cus=256) -> int:
    """Columns of a workgroup of the sweeps at K = 128."""
    rule = _lib.load_library()["_ZN3gdn18sweep_columns_k128Eiiiilbbi"]
    rule.restype, rule.argtypes = ctypes.c_int, [ctypes.c_int] * 4 + [ctypes.c_int64, ctypes.c_bool, ctypes.c_bool, ctypes.c_int]
    return rule(N, H, V, longest, chunks, packed, padded, cus)
