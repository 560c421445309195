"""Builds ``libmonarch_hip.so`` in-tree with hipcc for gfx950 (cross-compiles without a GPU) and, for the running interpreter
and its PyTorch, the native host path beside it."""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


def build(force: bool = True, jobs: int = 8) -> str:
    cmd = ["make", "-C", os.path.join(HERE, "csrc"), f"-j{jobs}", "all", "python", f"PYTHON={sys.executable}"]
    if force:
        cmd.append("-B")
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout)
        raise RuntimeError("building libmonarch_hip.so failed")
    return os.path.join(HERE, "libmonarch_hip.so")


if __name__ == "__main__":
    print(build())
