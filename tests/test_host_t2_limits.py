"""CPU: which grids the two-step kernel's 32-bit offsets reach (csrc/t2_limits.h).

A lane without cells uses the offset OOB = 2^32 - 16, which is out of range only
of arrays of at most that many bytes: the 3N FP32 values of 651 x 1661 x 331 cells
are 2^32 - 4 bytes.
"""

import shutil
import subprocess
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import pytest

import wakis_amd as wa

GRIDS = [(256, 256, 512), (651, 1661, 331), (651, 1661, 330), (710, 710, 710), (711, 710, 709),
         (560, 560, 570), (563, 564, 563), (564, 564, 564), (2, 2, 89_478_485),
         (2, 2, 44_739_242), (2, 2, 44_739_243), (11, 331, 98303)]


@pytest.fixture(scope="module")
def library_rule(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("t2")
    (d / "m.cpp").write_text('#include "t2_limits.h"\n#include <cstdio>\n#include <cstdlib>\n'
                             'int main(int n, char **v) { printf("%u %d", wf::OOB, '
                             "wf::t2_in_reach(atoll(v[1]), atoi(v[2]))); }\n")
    subprocess.run([cxx, "-std=c++17", "-I", str(Path(wa.__file__).parent / "csrc"),
                    str(d / "m.cpp"), "-o", str(d / "m")], check=True)

    def rule(n, elem):
        out = subprocess.run([str(d / "m"), str(n), str(elem)], check=True, capture_output=True,
                             text=True).stdout.split()
        return int(out[0]), bool(int(out[1]))
    return rule


@pytest.mark.parametrize("dims", GRIDS)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_no_array_reaches_the_offset_of_idle_lanes(library_rule, dims, dtype):
    x, y, z = dims
    elem = np.dtype(dtype).itemsize
    oob, ok = library_rule(x * y * z, elem)
    assert ok == (3 * x * y * z * elem <= oob)
    if ok:  # the metric tables, in one array
        assert 2 * (y * z + x * z + x * y) * elem <= oob
    assert wa.SolverFIT3D._pairs_in_reach(SimpleNamespace(N=x * y * z, dtype=dtype)) == ok


def test_the_grids_cover_both_sides(library_rule):
    assert not library_rule(651 * 1661 * 331, 4)[1] and library_rule(651 * 1661 * 330, 4)[1]
    assert 2 ** 32 - 16 < 12 * 651 * 1661 * 331 < 2 ** 32
