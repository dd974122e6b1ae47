"""Binding of libpikv_hip.so (the C ABI declared in include/pikv_hip.h): ctypes signatures, and call() through the typed entry
points of csrc/call.cpp.

The library is the only compute path of this package: if it is missing, or a
call returns a non-zero status, an exception is raised.  There is no CPU or
PyTorch fallback.  The reference's binding precedent is PiKVKernels.__init__
(core/single/pikv_kernels.py:36-52), which resolves the shared library next to
the package and silently falls back to torch when it is absent; here the
absence is an error.
"""
from __future__ import annotations

import ctypes as C
import os
import threading

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("PIKV_HIP_LIB", os.path.join(_HERE, "libpikv_hip.so"))

# element types / schemes / policies (mirrors include/pikv_hip.h)
F32, BF16 = 0, 1
Q_I8_SYM, Q_I8_ASYM, Q_I4_ASYM, Q_I4_SYM = 0, 1, 2, 3
EVICT_H2O, EVICT_LRU, EVICT_ALL = 0, 1, 2
SCORE_TILE = 64
MAX_PLANES = 10

_p, _i, _l, _f, _d = C.c_void_p, C.c_int, C.c_int64, C.c_float, C.c_double

# name -> (restype, argtypes)
SIGNATURES = {
    "pikv_status_string": (C.c_char_p, [_i]),
    "pikv_abi_version": (_i, []),
    "pikv_router_fused": (_i, [_p, _p, _i, _p, _p, _p, _f, _f, _i, _l, _i, _i, _i, _l,
                               _p, _p, _p, _p, _p, _p, _p, _l, _p]),
    "pikv_router_tail": (_i, [_p, _p, _p, _p, _p, _f, _f, _i, _i, _l, _i, _i, _l,
                              _p, _p, _p, _p, _p, _p, _l, _p]),
    "pikv_capacity_slots": (_i, [_p, _l, _i, _l, _p, _p, _p, _l, _p]),
    "pikv_capacity_slots_static": (_i, [_p, _l, _i, _l, _p, _p, _p]),
    "pikv_capacity_slots_static_max": (_l, []),
    "pikv_router_workspace_bytes": (_l, [_l, _i, _i]),
    "pikv_router_fused_workspace_bytes": (_l, [_l, _i, _i, _i]),
    "pikv_quant_scatter": (_i, [_p, _p, _i, _l, _i, _i, _i, _i, _p, _p, _p, _p, _p, _i,
                                _p, _p, _p, _p, _p, _p, _p, _p, _f, _p]),
    "pikv_cache_advance": (_i, [_p, _p, _p, _i, _l, _p]),
    "pikv_quant_gather": (_i, [_p, _p, _i, _i, _i, _i, _p, _p, _p, _l, _p, _p, _p, _p, _i,
                               _p, _p, _p, _p, _p, _p, _p, _p, _f, _p]),
    "pikv_quant_append": (_i, [_p, _p, _i, _l, _i, _i, _i, _p, _p, _p, _p, _i,
                               _p, _p, _p, _p, _p, _p, _p, _p, _f, _p]),
    "pikv_quantize_rows": (_i, [_p, _i, _l, _i, _i, _i, _l, _p, _p, _p, _p]),
    "pikv_quant8_minshift": (_i, [_p, _i, _l, _i, _p, _p, _p, _p, _p]),
    "pikv_gather_dequant": (_i, [_p, _p, _p, _i, _i, _i, _p, _l, _l, _p, _i, _p]),
    "pikv_gather_dequant_scores": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _p, _i, _f,
                                        _p, _p, _i, _l, _l, _p, _p, _p, _p]),
    "pikv_h2o_accumulate": (_i, [_p, _p, _p, _i, _p, _p, _i, _l, _l, _f, _f, _i,
                                 _p, _p, _p, _p, _p]),
    "pikv_attend_values": (_i, [_p, _p, _l, _p, _p, _p, _i, _i, _i, _i, _i, _p, _p, _i, _l,
                                _f, _f, _p, _p, _p, _p, _l, _p]),
    "pikv_attend_workspace_bytes": (_l, [_i, _i, _i, _l]),
    "pikv_decode_attend": (_i, [_p, _p, _p, _p, _p, _p, _i, _i, _i, _i, _i, _p, _i, _f, _p, _p, _i, _l,
                                _f, _f, _p, _p, _p, _p, _l, _p]),
    "pikv_decode_attend_workspace_bytes": (_l, [_i, _i, _i, _l]),
    "pikv_prefill_attend": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _i, _f, _p, _p, _p, _p, _p, _p, _i, _i,
                                 _p, _p, _l, _p, _p, _l, _p]),
    "pikv_prefill_attend_workspace_bytes": (_l, [_i, _i, _i, _i, _i, _l]),
    "pikv_evict_select": (_i, [_i, _p, _p, _p, _p, _p, _p, _i, _l, _p, _p, _p, _p, _l, _p]),
    "pikv_evict_select_h2o": (_i, [_d, _d, _p, _p, _p, _p, _p, _p, _i, _l, _p, _p, _p, _p, _l, _p]),
    "pikv_evict_workspace_bytes": (_l, [_i, _l]),
    "pikv_h2o_budget": (_i, [_p, _i, _d, _d, _p, _p, _p]),
    "pikv_cache_make_room": (_i, [_i, _p, _l, _l, _d, _d, _i, _i, _p, _p, _p, _p, _p, _i, _l,
                                  C.POINTER(_p), C.POINTER(_l), _i, _p, _p, _p, _p, _p, _l, _p]),
    "pikv_compact_rows": (_i, [C.POINTER(_p), C.POINTER(_l), _i, _p, _p, _p, _p, _i, _p]),
    "pikv_linear_group": (_i, [_p, _l, _i, _i, C.POINTER(_p), C.POINTER(_p), C.POINTER(C.c_int32), C.POINTER(C.c_int32),
                               _i, C.POINTER(_p), C.POINTER(_p), C.POINTER(_f), C.POINTER(_p), _p, _l, _p]),
    "pikv_linear_group_workspace_bytes": (_l, [_l, _i, _i]),
    "pikv_linear_tiled": (_i, [_p, _l, _i, _i, C.POINTER(_p), C.POINTER(_p), C.POINTER(C.c_int32), C.POINTER(_p), _p]),
    "pikv_cache_mean": (_i, [_p, _p, _p, _i, _i, _i, _p, _p, _i, _l, _p, _p, _l, _p]),
    "pikv_cache_mean_workspace_bytes": (_l, [_i, _i, _l]),
    "pikv_value_lora": (_i, [_p, _i, _i, _i, C.POINTER(_p), C.POINTER(_p), C.POINTER(_f), _p, _p]),
    "pikv_expert_combine": (_i, [C.POINTER(_p), C.POINTER(_p), C.POINTER(_f), _p, _p, _l, _i, _i, _p, _p, _p]),
    "pikv_expert_combine_factors": (_i, [C.POINTER(_p), C.POINTER(_p), C.POINTER(_p), _i, C.POINTER(_f), _p, _p, _l, _i, _i,
                                         _p, _p, _p]),
    "pikv_adaptive_router": (_i, [_p, _i, _i, _i, _i, _i, _i, _p, _p, _p, _p, _p, _p, _p, _f, _p, _p, _p, _f, _p, _p, _p,
                                  _p, _f, _p, _p, _p, _p, _p, _p, _p, _p]),
    "pikv_quant_scatter_routed": (_i, [_p, _p, _l, _i, _i, _i, _i, _p, _p, _p, _p, _p, _i,
                                       _p, _p, _p, _p, _p, _p, _p, _p, _f, _p]),
    "pikv_fakequant_colblocks": (_i, [_p, _l, _i, _i, _i, _i, _p, _p, _p, _p, _l, _p]),
    "pikv_fakequant_workspace_bytes": (_l, [_l, _i, _i]),
    "pikv_fakequant_preset": (_i, [_p, _l, _i, _i, _i, _i, _p, _p, _p, _p, _l, _p]),
}

_lib = None
_lock = threading.Lock()


class PiKVNativeError(RuntimeError):
    """The native library is missing or returned an error status."""


def lib() -> C.CDLL:
    """Load libpikv_hip.so once; raise if it is not built."""
    global _lib
    if _lib is None:
        with _lock:
            if _lib is None:
                if not os.path.exists(LIB_PATH):
                    raise PiKVNativeError(
                        f"{LIB_PATH} not found: build it with `python -m pikv_amd.build` "
                        "(there is no CPU fallback)")
                handle = C.CDLL(LIB_PATH)
                for name, (res, args) in SIGNATURES.items():
                    fn = getattr(handle, name)
                    fn.restype = res
                    fn.argtypes = args
                _lib = handle
    return _lib


def status_string(code: int) -> str:
    return lib().pikv_status_string(int(code)).decode()


def check(code: int, what: str) -> None:
    if code != 0:
        raise PiKVNativeError(f"{what} failed: {status_string(code)} (status {code})")


try:
    from . import _call
except ImportError as e:                 # not built, or it does not load: whoever needs it is told
    _call, _call_error = None, e
_entries = _of_checked = None


def entry_module():
    """The extension module of csrc/call.cpp."""
    if _call is None:
        raise PiKVNativeError(f"pikv_amd/_call is not built or does not load ({_call_error}): build it with "
                              "`python -m pikv_amd.build`") from _call_error
    return _call


def entries():
    """The module of typed entry points (csrc/call.cpp), bound to the library that lib() loads.  Every call of this package
    goes through it; lib() remains for a ctypes caller."""
    global _entries, _of_checked
    if _entries is None:
        lib()
        with _lock:
            if _entries is None:
                module = entry_module()
                try:
                    module.load(LIB_PATH)
                except OSError as e:
                    raise PiKVNativeError(f"{e}: build both with `python -m pikv_amd.build`") from e
                _of_checked = module.of_checked
                _entries = module
    return _entries


def call(name: str, *args) -> None:
    """Call an int-status entry point and raise on a non-zero status.  Pointers: GPU tensors, addresses, None; lists for host arrays."""
    code = getattr(_entries or entries(), name)(*args)
    if code:
        check(code, name)


def launch(name: str, *args) -> None:
    """call() for a caller that has seen that its tensors are on the GPU."""
    code = getattr(_of_checked or entries().of_checked, name)(*args)
    if code:
        check(code, name)


def size(name: str, *args) -> int:
    """Call an entry point that returns a number of bytes."""
    return getattr(_entries or entries(), name)(*args)
