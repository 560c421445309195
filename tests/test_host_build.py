"""What the Makefile and the package's build step build, and for whom.  No GPU; nothing is compiled here."""
import os
import struct
import subprocess
import sys
import sysconfig

import monarch_amd.build
from monarch_amd import _native

CSRC = os.path.join(os.path.dirname(monarch_amd.build.__file__), "csrc")


def plan(*args):
    return subprocess.run(["make", "-n", "-B", "-C", CSRC, *args], capture_output=True, text=True)


def test_the_library_alone_needs_no_python():
    # the build of a C or Rust program: no interpreter is asked and no extension is built
    p = plan("PYTHON=/no/such/python")
    assert p.returncode == 0 and "libmonarch_hip.so" in p.stdout and "host_calls" not in p.stdout and "python" not in p.stderr


def test_the_extension_is_built_for_the_interpreter_that_builds_it(monkeypatch):
    commands = []

    class Done:
        returncode, stdout = 0, ""

    monkeypatch.setattr(subprocess, "run", lambda cmd, **kw: commands.append(cmd) or Done)
    monarch_amd.build.build()
    monkeypatch.undo()
    args = commands[0][1:]
    assert f"PYTHON={sys.executable}" in args
    suffix = sysconfig.get_config_var("EXT_SUFFIX")
    assert "cpython" in suffix
    p = subprocess.run(["make", "-n", *args], capture_output=True, text=True)
    assert p.returncode == 0 and f"-o ../_host_calls{suffix} " in p.stdout and f"-I{sysconfig.get_paths()['include']} " in p.stdout
    assert _native.host.slice_copy.__self__.__file__.endswith("/_host_calls" + suffix)


def test_an_interpreter_without_pytorch_is_named():
    p = plan("python", "PYTHON=/bin/false")
    assert p.returncode != 0 and "/bin/false is no Python with PyTorch" in p.stderr


def test_the_extension_has_no_thread_local_data():
    # it would slow down every thread-local access of a thread, a launch's among them, where the library was loaded first
    with open(_native.host.slice_copy.__self__.__file__, "rb") as f:
        elf = f.read()
    start, size, count = struct.unpack_from("<Q", elf, 32)[0], *struct.unpack_from("<HH", elf, 54)
    kinds = [struct.unpack_from("<I", elf, start + k * size)[0] for k in range(count)]
    assert 1 in kinds and 7 not in kinds  # PT_LOAD, PT_TLS
