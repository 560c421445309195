"""The native host path (``csrc/host_calls.cpp``): the checks of a call on plain tensors and the call into the library,
without a Python statement per check.

Every function of ``host`` returns the library's status, or ``NOT_TAKEN`` for a call that is not one on plain tensors or
that does not pass a check; the Python code behind it then runs as it would without it.  Without the built extension the
first call raises ``MonarchHipNotBuilt``, as without the library.
"""
from __future__ import annotations

import torch  # noqa: F401  (its libraries have to be in the process before the extension that uses them)

from ._lib import MonarchHipNotBuilt
from .ndslice import Slice

try:
    from . import _host_calls as host

    host.set_slice_type(Slice)
except ImportError as e:
    _reason = str(e)

    class _NotBuilt:
        def __getattr__(self, name):
            raise MonarchHipNotBuilt(f"the native host path is missing ({_reason}): build it with `python -m monarch_amd.build`")

    host = _NotBuilt()
