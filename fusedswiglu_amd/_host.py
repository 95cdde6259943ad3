"""The native host path (csrc/fsw_host.cpp): checks, allocations, launches and autograd nodes of calls that nothing watches.

`swiglu(x, w_gate, w_up, dtype_code, recompute, weights_out_in, operator)` (w_up None: w_gate is a packed weight; dtype_code -1:
either type; operator: a backward pass that is watched or recorded goes through the custom operator) and `down_proj(act, w_down,
weights_out_in)` give the result, with an autograd node behind it where a gradient is recorded, or None for every call that is
not plain: the caller then takes the general path, which also raises the errors.

Where the extension is not there or does not load (it is tied to the torch it was built with; the kernels' library is not), every call
takes the general path on the same kernels, after one warning."""
from __future__ import annotations

import importlib.machinery
import importlib.util
import os
import threading
import warnings

from . import _abi

PATH = os.path.join(os.path.dirname(_abi.LIBRARY_PATH), "_fsw_host.so")

_module = None
_lock = threading.Lock()


class _General:
    """In the extension's place where it cannot be used"""

    @staticmethod
    def swiglu(*_):
        return None

    down_proj = swiglu


def _import_extension():
    import torch  # (its libraries come first)

    from . import ops
    from .kernels import _launch

    loader = importlib.machinery.ExtensionFileLoader("_fsw_host", PATH)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_fsw_host", PATH, loader=loader))
    loader.exec_module(module)
    if module.torch_version != torch.__version__.split("+")[0]:
        raise ImportError(f"built with torch {module.torch_version}, this is {torch.__version__}")
    module.setup(_abi.check, ops._general_backward, ops._general_down_backward, _launch._PAD_MIN_WORK,
                 _launch._PAD_MIN_WORK // _launch._PAD_MIN_STEPS_SHARE, _launch._TILED_MAX_LD)
    return module


def load():
    """The extension module, or what answers None to every call."""
    global _module
    if _module is not None:
        return _module
    with _lock:
        if _module is None:
            try:
                _abi.lib()
            except _abi.LibraryNotBuiltError:
                return _General  # (the general path says so, if it comes to the library; not kept: it may be built yet)
            try:
                _module = _import_extension()
            except Exception as e:  # whatever keeps it from loading, the general path needs nothing of it
                warnings.warn(f"{PATH} cannot be used ({e}): calls take the slower Python host path; build it with "
                              f"`make -C {os.path.dirname(PATH)}`", RuntimeWarning, stacklevel=4)
                _module = _General
    return _module


def swiglu(x, w_gate, w_up, dtype_code=-1, recompute=False, weights_out_in=False, operator=False):
    return (_module or load()).swiglu(x, w_gate, w_up, dtype_code, recompute, weights_out_in, operator)


def down_proj(act, w_down, weights_out_in):
    return (_module or load()).down_proj(act, w_down, weights_out_in)
