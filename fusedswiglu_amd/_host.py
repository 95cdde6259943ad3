"""The native host path (csrc/fsw_host.cpp): checks, allocations, launches and autograd nodes of calls that nothing watches.

`swiglu(x, w_gate, w_up, dtype_code, recompute, weights_out_in, operator)` (w_up None: w_gate is a packed weight; dtype_code -1:
either type; operator: a backward pass that is watched or recorded goes through the custom operator) and `down_proj(act, w_down,
weights_out_in)` give the result, with an autograd node behind it where a gradient is recorded, or None for every call that is
not plain: the caller then takes the general path, which also raises the errors."""
from __future__ import annotations

import importlib.machinery
import importlib.util
import os
import threading

from . import _abi

PATH = os.path.join(os.path.dirname(_abi.LIBRARY_PATH), "_fsw_host.so")

_module = None
_lock = threading.Lock()


def load():
    """The extension module.  Raises LibraryNotBuiltError if it was not built."""
    global _module
    if _module is not None:
        return _module
    with _lock:
        if _module is None:
            if not os.path.exists(PATH):
                raise _abi.LibraryNotBuiltError(f"{PATH} not found; build it with `make -C {os.path.dirname(PATH)}`")
            import torch  # noqa: F401  (its libraries come first)

            from . import ops
            from .kernels import _launch

            _abi.lib()
            loader = importlib.machinery.ExtensionFileLoader("_fsw_host", PATH)
            module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_fsw_host", PATH, loader=loader))
            loader.exec_module(module)
            module.setup(_abi.check, ops._general_backward, ops._general_down_backward, _launch._PAD_MIN_WORK,
                         _launch._PAD_MIN_WORK // _launch._PAD_MIN_STEPS_SHARE, _launch._TILED_MAX_LD)
            _module = module
    return _module


def swiglu(x, w_gate, w_up, dtype_code=-1, recompute=False, weights_out_in=False, operator=False):
    return (_module or load()).swiglu(x, w_gate, w_up, dtype_code, recompute, weights_out_in, operator)


def down_proj(act, w_down, weights_out_in):
    return (_module or load()).down_proj(act, w_down, weights_out_in)
