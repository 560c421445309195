"""The native host path (``csrc/host_calls.cpp``): the checks of a call on plain tensors and the call into the library,
without a Python statement per check.

Every function of ``host`` returns the library's status, or ``NOT_TAKEN`` for a call that is not one on plain tensors or
that does not pass a check; the Python code behind it then runs as it would without it.

The extension is loaded by the first call, not by an import, and ``lib()`` before it: the library reads its environment while it
is loaded.  Without the extension that call raises ``MonarchHipNotBuilt``, as without the library.
"""
from __future__ import annotations

import torch  # noqa: F401  (its libraries have to be in the process before the extension that uses them)

from . import _lib
from .ndslice import Slice

_NAMES = ("slice_copy", "slice_copy_many", "rdma_copy", "transfer_many", "reduce", "stack", "reduce_scatter", "flat_copy", "quantize_bucket",
          "dequant_accumulate_bucket", "tensor_addresses", "NOT_TAKEN")


def extension():
    """The extension module."""
    _lib.lib()
    try:
        from . import _host_calls
    except ImportError as e:
        raise _lib.MonarchHipNotBuilt(f"the native host path is missing ({e}): build it with `python -m monarch_amd.build`") from e
    _host_calls.set_slice_type(Slice)
    return _host_calls


class _Host:
    """The extension's functions, once one of them has been asked for."""

    def __getattr__(self, name):
        if name not in _NAMES:
            raise AttributeError(name)
        ext = extension()
        self.__dict__.update((n, getattr(ext, n)) for n in _NAMES)
        return self.__dict__[name]


host = _Host()
