"""When the native host path and the library behind it are loaded, and which library it is.  Each case in a process of its own,
on the CPU: calls on CPU tensors end in the checks behind the native path."""
import os
import shutil
import subprocess
import sys

from monarch_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
COMMON = f"""
import sys, warnings
sys.path.insert(0, {ROOT!r})
import torch
from monarch_amd import MhipError, MonarchHipNotBuilt, Slice, _lib, fp8, reduce as R, staging
def mapped(name):
    return [line.split()[-1] for line in open("/proc/self/maps") if name in line]
def error(call, *args):
    try:
        call(*args)
    except Exception as e:
        return type(e).__name__ + " " + str(getattr(e, "name", ""))
x = torch.zeros(8)
"""


def run(code):
    p = subprocess.run([sys.executable, "-c", COMMON + code], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-2000:]
    return p.stderr


def test_an_import_loads_no_library():
    # the library reads its environment while it is loaded, so that happens with the first call
    run("""
assert not mapped("libmonarch_hip") and not mapped("_host_calls")
assert error(R.all_reduce, x, [x], 0) == "MhipError InvalidDevice"
assert mapped("libmonarch_hip") and mapped("_host_calls")
""")


def test_a_missing_library_is_an_error_of_every_call(tmp_path):
    run(f"""
s = Slice(offset=0, sizes=[8], strides=[1])
_lib._lib, _lib.LIB_PATH = None, {str(tmp_path / "libmonarch_hip.so")!r}
for call, args in ((staging.pack, (x, s, x)), (staging.unpack, (x, s, x)), (R.all_reduce, (x, [x], 0)), (staging.transfer_many, ([1], [1], [1]))):
    assert error(call, *args).startswith("MonarchHipNotBuilt"), call
""")


def test_calls_of_another_library_do_not_reach_the_one_beside_the_extension(tmp_path):
    other = str(tmp_path / "libmonarch_hip.so")
    shutil.copy(_lib.LIB_PATH, other)
    run(f"""
_lib.LIB_PATH = {other!r}
s = Slice(offset=0, sizes=[8], strides=[1])
assert error(staging.pack, x, s, x) == "MhipError InvalidDevice" and error(R.all_reduce, x, [x], 0) == "MhipError InvalidDevice"
assert set(mapped("libmonarch_hip")) == {{{other!r}}} and not mapped("_host_calls")
assert staging.host.slice_copy(True, x, s, x) == staging.host.NOT_TAKEN and staging.host.tensor_addresses([x], b"", x) is None
""")


def test_without_the_extension_calls_take_the_ctypes_path():
    for state in ("sys.modules['monarch_amd._host_calls'] = None", "from monarch_amd import _host_calls; _host_calls.TORCH_VERSION = '1.2.3'"):
        err = run(f"""
{state}
s = Slice(offset=0, sizes=[8], strides=[1])
for _ in range(2):
    for call, args in ((staging.pack, (x, s, x)), (staging.unpack, (x, s, x)), (R.all_reduce, (x, [x], 0)), (fp8.quantize, (x,))):
        assert error(call, *args) == "MhipError InvalidDevice", call
assert staging.host.slice_copy(True, x, s, x) == staging.host.NOT_TAKEN
""")
        assert err.count("no native host path") == 1
