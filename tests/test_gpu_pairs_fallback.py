"""GPU: calls that ask for two steps per launch where the kernel does not apply run
one step per launch, with the same results and the caller's arguments as they were:
rows for which no tile fits a workgroup, and coefficients read from arrays."""

import numpy as np
import pytest

from tests.test_gpu_two_step import _beam_setup, _cavity_solver

pytestmark = pytest.mark.gpu


def _run(dims, dtype, two_step, codes=True):
    s = _cavity_solver(dims, two_step, 0, dtype)
    s.use_material_code = codes
    args, cap = _beam_setup(s, 7)
    for n0, k in ((0, 4), (4, 3)):
        a = args(n0, k)
        s._run(a)
        assert s.last_path == "fused" and not s.last_pairs and not s.last_two_step
        assert a.two_step == two_step
    return [s.E.to_numpy(), s.H.to_numpy(), s.J.to_numpy(), cap.cpu().numpy()]


# 64 tiles of the longest row that a workgroup holds with its halo: 38,656 cells
# FP32, 19,328 FP64
@pytest.mark.parametrize("dims,dtype,codes", [((38800, 6, 6), np.float32, True),
                                              ((19400, 6, 6), np.float64, True),
                                              ((64, 20, 24), np.float32, False),
                                              ((64, 20, 24), np.float64, False)])
@pytest.mark.parametrize("two_step", [1, 8])
def test_single_steps_where_pairs_do_not_apply(dims, dtype, codes, two_step):
    print("pairs fallback", dims, np.dtype(dtype).name, codes, two_step, flush=True)
    ref = _run(dims, dtype, 0, codes)
    got = _run(dims, dtype, two_step, codes)
    assert ref[0].any()
    for name, r, g in zip(("E", "H", "J", "capture"), ref, got):
        assert np.array_equal(g, r), name
