"""GPU: what emsolve with a plane wave raises where a source value passes the FP32
range during the run (FP32 fields, an FP64 time step, so FP64 source values): the
error of the step-by-step loop, at the same step."""

import numpy as np
import pytest

from tests.test_gpu_emsolve_source import _solver

pytestmark = pytest.mark.gpu

DIMS = (12, 9, 44)


def _rising(wa, dtype):
    # E_x = 18 A cos(w t + phase): about 0 at first, past 3.4e38 within a period
    return wa.PlaneWave(f=1e9, zs=5, amplitude=5e37 if dtype == np.float32 else 1e300,
                        phase=-0.5 * np.pi)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_source_value_past_the_storage_type(dtype):
    import wakis_amd as wa
    print("emsolve overflow", np.dtype(dtype).name, flush=True)
    steps = []
    for by_step in (True, False):
        s = _solver(DIMS, dtype, "pml", "pec")
        s.dt = np.float64(s.dt)
        n = int(0.3e-9 / float(s.dt))
        kw = dict(source=_rising(wa, dtype), callback=(lambda *_: None) if by_step else None)
        if dtype == np.float32:
            with pytest.raises(RuntimeError, match="overflow"):
                s.emsolve(n, **kw)
        else:
            s.emsolve(n, **kw)
        steps.append(s.nstep)
    assert steps[0] == steps[1] > 3
