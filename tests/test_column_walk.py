"""The column kernels look up only the pixels of their lists, and no index
leaves the pair table.  Compiles the walk that the kernels run
(multigpugridder_amd/csrc/mgg_columns.h) for the host."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def walker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("col") / "column_walk")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(HERE, "..", "multigpugridder_amd", "csrc"), "-o", exe,
                    os.path.join(HERE, "column_walk.cpp")], check=True)
    return lambda what: [line.split() for line in subprocess.run(
        [exe, what], check=True, capture_output=True, text=True).stdout.strip().splitlines()]


def test_each_pixel_of_a_row_once_and_no_other(walker):
    rows = walker("rows")
    assert len(rows) == 17
    for cnt, *seen in rows:
        assert sorted(map(int, seen)) == list(range(int(cnt)))


def test_no_index_leaves_the_table(walker):
    rows = walker("range")
    # back projection with 5 and 6 slots, the transpose with 6, 8 and 10; both ends
    assert sorted((int(r[0]), int(r[1]), int(r[2])) for r in rows) == sorted(
        (m, k, s) for m, ks in ((0, (5, 6)), (1, (6, 8, 10))) for k in ks for s in (-1, 1))
    for mode, slots, sign, index, lo, hi in rows:
        # 4 entries for the kernel's FP32 positions and frames off by 5e-3
        assert int(lo) + 4 <= float(index) <= int(hi) - 1 - 4, (mode, slots, sign, index)
