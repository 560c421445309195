"""Run by test_gpu_host_calls.py in a process of its own, with a folder that holds a copy of the extension beside the library of
c_abi/held_library.c: while the library runs without the interpreter's lock, all lists of the call are emptied, and their
tensors have to live on until the call returns, and no longer."""
import ctypes
import importlib.util
import os
import sys
import weakref

import torch

folder = sys.argv[1]
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
name = next(f for f in os.listdir(folder) if f.startswith("_host_calls"))
spec = importlib.util.spec_from_file_location("_host_calls", os.path.join(folder, name))
ext = importlib.util.module_from_spec(spec)
library = ctypes.CDLL(os.path.join(folder, "libmonarch_hip.so"))

from monarch_amd import Slice  # noqa: E402  (its library has the same name: the extension's goes first)

ext.set_slice_type(Slice)
DEV = "cuda:0"


def tensors(n, numel, dtype=torch.float32):
    return [torch.zeros(numel, dtype=dtype, device=DEV) for _ in range(n)]


def run(call, *args, status=0):
    lists = [a for a in args if isinstance(a, list)]
    refs = [weakref.ref(t) for a in lists for t in a if isinstance(t, torch.Tensor)]
    alive = []

    def hook():
        for a in lists:
            a.clear()
        alive.append([r() is not None for r in refs])
        return status

    callback = ctypes.CFUNCTYPE(ctypes.c_int)(hook)
    ctypes.c_void_p.in_dll(library, "hook").value = ctypes.cast(callback, ctypes.c_void_p).value
    got = getattr(ext, call)(*args)
    assert len(alive) == 1 and all(alive[0]), (call, alive)
    assert all(r() is None for r in refs), call
    print(call, "held", len(refs), flush=True)
    return got


out, flat = torch.zeros(64, device=DEV), torch.zeros(320, device=DEV)
views = lambda: [Slice(offset=8 * k, sizes=[8], strides=[1]) for k in range(5)]
table = torch.zeros(3, dtype=torch.int64, device=DEV)
offsets = torch.zeros(4, dtype=torch.int64, device=DEV)
assert run("reduce", out, tensors(5, 64), 0) == 0
assert run("stack", flat, tensors(5, 64)) == 0
assert run("reduce_scatter", tensors(5, 8), views(), tensors(8, 64), Slice(offset=0, sizes=[64], strides=[1]), 0) == 0
assert run("slice_copy_many", True, flat, views(), tensors(5, 8)) == 0
assert run("slice_copy_many", False, flat, views(), tensors(5, 8), status=7) == 7
assert run("dequant_accumulate_bucket", table, offsets, 2000, None, tensors(6, 2000, torch.uint8), tensors(6, 2)) == 0
# a status of 1 is not the mark of a call that was left alone
assert run("transfer_many", [16], [32], [8], 0, status=1) == -1 != ext.NOT_TAKEN
print("host_calls_held ok")
