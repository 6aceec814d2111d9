"""CPU: which grids the two-step kernel's 32-bit offsets reach (csrc/t2_limits.h).

A lane without cells uses the offset OOB = 2^32 - 16, which is out of range only
of arrays of at most that many bytes: 3N values of 2^32 - 4 bytes (FP32, 651 x 1661
x 331 cells) or a metric table longer than the fields (a line of cells) are not.
"""

import shutil
import subprocess
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import pytest

import wakis_amd as wa

CSRC = Path(wa.__file__).parent / "csrc"
GRIDS = [(256, 256, 512), (651, 1661, 331), (651, 1661, 330), (710, 710, 710), (711, 710, 709),
         (560, 560, 570), (563, 564, 563), (564, 564, 564), (1, 1, 200_000_000),
         (1, 1, 300_000_000), (1, 2, 120_000_000), (2, 1, 150_000_000), (2, 2, 89_478_485),
         (1, 17895697, 20), (11, 331, 98303)]


def _arrays(dims, elem):
    x, y, z = dims
    return elem * 3 * x * y * z, elem * 2 * (y * z + x * z + x * y)


@pytest.fixture(scope="module")
def library_rule(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("t2")
    (d / "m.cpp").write_text('#include "t2_limits.h"\n#include <cstdio>\n#include <cstdlib>\n'
                             "int main(int n, char **v) { printf(\"%u %d\", wf::OOB, "
                             "wf::t2_in_reach(atoll(v[1]), atoll(v[2]), atoll(v[3]), "
                             "atoi(v[4]))); }\n")
    subprocess.run([cxx, "-std=c++17", "-I", str(CSRC), str(d / "m.cpp"), "-o", str(d / "m")],
                   check=True)

    def rule(dims, elem):
        out = subprocess.run([str(d / "m"), *map(str, dims), str(elem)], check=True,
                             capture_output=True, text=True).stdout.split()
        return int(out[0]), bool(int(out[1]))
    return rule


@pytest.mark.parametrize("dims", GRIDS)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_no_array_reaches_the_offset_of_idle_lanes(library_rule, dims, dtype):
    elem = np.dtype(dtype).itemsize
    oob, ok = library_rule(dims, elem)
    assert ok == all(n <= oob for n in _arrays(dims, elem))
    s = SimpleNamespace(Nx=dims[0], Ny=dims[1], Nz=dims[2], N=dims[0] * dims[1] * dims[2],
                        dtype=dtype)
    assert wa.SolverFIT3D._pairs_in_reach(s) == ok


def test_the_grids_cover_both_sides(library_rule):
    got = {(d, e): library_rule(d, e)[1] for d in GRIDS for e in (4, 8)}
    assert not got[(651, 1661, 331), 4] and got[(651, 1661, 330), 4]
    # 3N within 4 GiB, the metric table not
    assert _arrays((1, 1, 300_000_000), 4)[0] < 2 ** 32 and not got[(1, 1, 300_000_000), 4]
