"""Which kernels a copy launches, without a GPU: tests/c_abi/launches.c links the library and takes the place of
``hipLaunchKernel``, so that sizes no GPU holds can be asked for."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIMIT = (1 << 31) - 1  # dividends of the kernels' divisions by multiplication stay below this


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("launches") / "launches")
    lib = os.path.join(ROOT, "monarch_amd")
    subprocess.check_call(["gcc", "-std=gnu11", "-O1", "-Wall", "-Wextra", "-Werror", "-rdynamic", "-I", os.path.join(ROOT, "include"),
                           os.path.join(ROOT, "tests", "c_abi", "launches.c"), "-o", exe, "-L", lib, "-lmonarch_hip", "-Wl,-rpath," + lib, "-ldl"])

    def run(pack, size, sizes, strides):
        line = " ".join(str(x) for x in (int(pack), size, 0, len(sizes), *sizes, *strides))
        out = subprocess.run([exe], input=line + "\n", capture_output=True, text=True, check=True, timeout=60).stdout.split()
        assert out[0] == "0", out
        return [(int(out[k]), out[k + 1]) for k in range(1, len(out), 2)]
    return run


@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("size,a,b", [(2, 8, 8), (2, 8, 9), (2, 9, 8), (1, 16, 16), (1, 16, 17), (4, 8, 8), (4, 4 * 33, 8), (8, 8, 17), (2, 65, 8), (2, 8, 65),
                                      (2, 520, 8)])
def test_tile_numbers_of_small_matrices_fit_their_divisions(launches, pack, size, a, b):
    # [n1, n2, a, b] -> [n1, n2, b, a] with a gap after every n2 matrices, up to 2^32 tiles and more: the transposing kernel of small
    # matrices is launched with fewer workgroups than its divisions take, whatever its tile; beyond that another kernel is
    def narrow(n):
        n1 = 1 << 12
        n2 = -(-n // n1)
        got = launches(pack, size, [n1, n2, b, a], [(n2 + 1) * a * b, a * b, 1, b])
        assert got
        return n1 * n2, sum(wg for wg, name in got if "slice_transpose_narrow_kernel" in name)

    n, wgs = narrow(1 << 24)
    per_matrix = round(wgs / n)
    assert per_matrix >= 1 and wgs >= n * per_matrix
    n, wgs = narrow((LIMIT - (1 << 20)) // per_matrix)
    assert n * per_matrix <= wgs < LIMIT
    for tiles in (LIMIT - 7, LIMIT + 2, 3 << 30, (1 << 32) - (1 << 13), 1 << 32, (1 << 32) + 100, 3 << 32):
        n, wgs = narrow(-(-tiles // per_matrix))
        assert n * per_matrix >= LIMIT - 8 and wgs == 0, tiles


@pytest.mark.parametrize("pack", [True, False])
def test_lanes_of_two_byte_transposes_follow_the_number_of_tiles(launches, pack):
    # tiles of 128 x 128 elements whose written rows are whole lines: 1024 lanes from eight tiles along both sides on, else 512; rows
    # that are not whole lines always 1024
    def kernel(rows, cols):
        got = launches(pack, 2, [cols, rows], [1, cols])
        return got[0][1]

    for tiles, lanes in ((5, 512), (7, 512), (8, 1024), (9, 1024)):
        for rows, cols in ((tiles * 128, 20096), (20096, tiles * 128)):
            assert f"slice_transpose_vec_kernelItLi{lanes}E" in kernel(rows, cols), (rows, cols)
        assert "slice_transpose_lines_kernelItLi1024E" in (kernel(tiles * 128 - 20, 20096) if pack else kernel(20096, tiles * 128 - 20))


@pytest.mark.parametrize("pack", [True, False])
def test_byte_matrices_of_many_tiles_take_the_general_addresses(launches, pack):
    # up to 768 tiles of 128 x 128 the short form (the parameter before the last), above it the general one and the columns of a
    # tile before its first store (the last one), above 23 MiB the general one in tiles of 256 x 256
    def forms(rows, cols):
        return {name.split("slice_transpose_narrow_kernelI")[1].split("EEEv")[0] for _, name in launches(pack, 1, [cols, rows], [1, cols])
                if "slice_transpose_narrow_kernel" in name}

    p = int(pack)
    for rows, cols in ((600, 600), (3001, 4001), (2047, 6101), (6141, 2001)):
        assert forms(rows, cols) == {f"hLi256ELb{p}ELi128ELi128ELb1ELb0"}
    for rows, cols in ((3073, 4001), (1025, 11001), (2049, 6001), (3301, 4001), (4801, 5001)):
        assert forms(rows, cols) == {f"hLi256ELb{p}ELi128ELi128ELb0ELb1"}
    for rows, cols in ((1672, 15051), (6301, 6501)):
        assert forms(rows, cols) == {f"hLi512ELb{p}ELi256ELi256ELb0ELb0"}
    assert not forms(6501, 6501)
