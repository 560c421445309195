"""The native host path (``csrc/host_calls.cpp``): the checks of a call on plain tensors and the call into the library,
without a Python statement per check.

Every function of ``host`` returns the library's status, or ``NOT_TAKEN`` for a call that is not one on plain tensors or
that does not pass a check; the Python code behind it then runs as it would without it.

The extension is loaded by the first call, not by an import, and ``lib()`` before it: the library reads its environment while it
is loaded, and a missing library is an error.  The extension is linked to the ``libmonarch_hip.so`` beside it.  Where ``lib()`` is
another one (``_lib.LIB_PATH``), or where the extension is missing or built for another PyTorch (a warning says so once), every
call is left alone and takes the ctypes path: the same kernels, 1.3 to 3.5 us more of host time.
"""
from __future__ import annotations

import os
import re
import warnings

import torch

from . import _lib
from .ndslice import Slice

NOT_TAKEN = -(1 << 63)
_CALLS = ("slice_copy", "slice_copy_many", "rdma_copy", "transfer_many", "reduce", "stack", "reduce_scatter", "flat_copy", "quantize_bucket",
          "dequant_accumulate_bucket")


def _release(version: str) -> str:
    return re.match(r"[0-9.]*[0-9]", version).group()


def extension():
    """The extension module, or None where calls have to take the ctypes path."""
    beside = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libmonarch_hip.so")
    if os.path.realpath(_lib.lib()._name) != os.path.realpath(beside):
        return None
    try:
        from . import _host_calls
    except ImportError as e:
        reason = str(e)
    else:
        if _release(_host_calls.TORCH_VERSION) == _release(torch.__version__):
            _host_calls.set_slice_type(Slice)
            return _host_calls
        reason = f"built for PyTorch {_host_calls.TORCH_VERSION}, this is {torch.__version__}"
    warnings.warn(f"calls take the ctypes path: no native host path ({reason}); build it with `python -m monarch_amd.build`",
                  RuntimeWarning, stacklevel=4)
    return None


class _Loaded:
    """Attributes without a hook: 45 ns a look-up against 64."""


class _Host:
    """The extension's functions, once one of them has been asked for."""

    def __getattr__(self, name):
        if name not in _CALLS and name not in ("tensor_addresses", "NOT_TAKEN"):
            raise AttributeError(name)
        ext = extension()
        if ext is not None:
            found = {n: getattr(ext, n) for n in (*_CALLS, "tensor_addresses", "NOT_TAKEN")}
        else:
            found = {n: lambda *args: NOT_TAKEN for n in _CALLS}
            found.update(tensor_addresses=lambda *args: None, NOT_TAKEN=NOT_TAKEN)
        self.__dict__.update(found)
        self.__class__ = _Loaded
        return found[name]


host = _Host()
