"""The copy planner's rules on views that move unit by unit (plan.cpp, plain C++): which of them stream past the caches
and which are gathered chunk by chunk.  Compiled with the host compiler, no GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MIB = 1 << 20


@pytest.fixture(scope="module")
def decide(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("plan") / "plan_rules")
    csrc = os.path.join(ROOT, "monarch_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", os.path.join(ROOT, "tests", "c_abi", "plan_rules.cpp"),
                    os.path.join(csrc, "plan.cpp"), "-o", exe], check=True)

    def run(elem_size, sizes, strides):
        line = " ".join(str(x) for x in (elem_size, 0, len(sizes), *sizes, *strides))
        out = subprocess.run([exe], input=line + "\n", capture_output=True, text=True, check=True).stdout.split()
        return tuple(int(x) for x in out)
    return run


@pytest.mark.parametrize("es", [1, 2, 4, 8])
@pytest.mark.parametrize("k", [2, 4])
def test_every_kth_element_streams_from_92_mib_of_lines_on(decide, es, k):
    cols = 4096
    rows = 92 * MIB // (cols * k * es)
    assert decide(es, [rows, cols], [cols * k, k]) == (es, 1, 0)
    assert decide(es, [rows - 1, cols], [cols * k, k]) == (es, 0, 0)
    assert decide(es, [32 * MIB // (cols * k * es), cols], [cols * k, k]) == (es, 0, 0)
    # every other row as well: the lines in between are not touched
    assert decide(es, [rows, cols], [2 * cols * k, k]) == (es, 1, 0)
    assert decide(es, [rows // 2, cols], [2 * cols * k, k]) == (es, 0, 0)


@pytest.mark.parametrize("nbytes", [8_000_000, 24_000_000, 400_000_000])
def test_interleaved_views_keep_to_the_cache(decide, nbytes):
    # the columns of a tall matrix and the channels of images packed side by side: every line holds units of all of them
    for es, k in ((4, 3), (4, 7), (2, 3), (1, 9), (8, 3), (8, 5)):
        n = nbytes // (k * es)
        assert decide(es, [k, n], [1, k])[1] == 0                       # [n, k].t()
        assert decide(es, [n, k], [1, n])[1] == 0                       # [k, n].t()
        b = nbytes // (50176 * k * es)
        assert decide(es, [b, k, 50176], [50176 * k, 1, k])[1] == 0     # [b, hw, k] -> [b, k, hw]
        assert decide(es, [b, 50176, k], [50176 * k, 1, 50176])[1] == 0


def test_units_far_apart_count_one_line_each(decide):
    # a stride of 1 KiB touches one line of 128 bytes per element, not 1 KiB
    assert decide(4, [92 * MIB // 128], [256]) == (4, 1, 0)
    assert decide(4, [92 * MIB // 128 - 1], [256]) == (4, 0, 0)


@pytest.mark.parametrize("es", [1, 2])
def test_four_to_seven_planes_are_gathered_from_6_mib_on(decide, es):
    for k in (4, 5, 6, 7):
        n = -(-6 * MIB // (k * es)) | 1   # odd, so that the unit stays the element
        assert decide(es, [n, k], [1, n]) == (es, 0, 1)
        assert decide(es, [n - 2 * k, k], [1, n - 2 * k])[2] == 0
        assert decide(es, [k, n], [1, k])[2] == 0      # the other way round
    for k in (2, 3):
        assert decide(es, [8 * MIB, k], [1, 8 * MIB + 1])[2] == 0
