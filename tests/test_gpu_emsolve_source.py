"""GPU: emsolve with a plane wave whose steps run in the library's loop
(wf_step_args.src_E, src_H, abc_low) against a step-by-step loop of
PlaneWave.update, one_step and wf_abc_low: E, H, J bitwise the same, for planes
and boxes on and off the faces, sources that end during the run, calls one after
another, FP32 and FP64; other sources and callers keep the step-by-step loop.
"""

import numpy as np
import pytest
from scipy.constants import c as c_light

pytestmark = pytest.mark.gpu


def _solver(dims, dtype, top, low, conductive=False):
    import wakis_amd as wa
    x, y, z = (np.linspace(0, 0.8e-3 * n, n + 1) for n in dims)
    grid = wa.GridFIT3D(x=x, y=y, z=z, verbose=0)
    return wa.SolverFIT3D(grid, bc_low=["periodic", "periodic", low],
                          bc_high=["periodic", "periodic", top],
                          bg=[1.0, 1.0, 0.3] if conductive else [1.0, 1.0], dtype=dtype, verbose=0)


def _wave(dims, nodes, **kw):
    import wakis_amd as wa
    return wa.PlaneWave(f=9 * c_light / (dims[2] * 0.8e-3), amplitude=3.0, phase=0.4, nodes=nodes,
                        **kw)


def _state(s):
    return [F.to_numpy() for F in (s.E, s.H, s.J)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("top,low", [("pml", "pec"), ("abc", "abc")])
@pytest.mark.parametrize("dims,steps,kw", [
    ((12, 9, 44), (75, 40), dict(zs=5)),                 # chunks of 32, a second call
    ((65, 5, 41), (50,), dict(zs=0)),                    # the copied face itself
    ((13, 66, 40), (37,), dict(zs=-1, xs=slice(2, 11), ys=slice(3, 60))),
    ((8, 7, 45), (35,), dict(zs=slice(1, 4), xs=3, ys=slice(None))),
    ((12, 9, 44), (2, 3, 4), dict(zs=5)),                # shortest calls
])
def test_same_as_step_by_step(dtype, top, low, dims, steps, kw):
    print("emsolve source", np.dtype(dtype).name, top, dims, steps, kw, flush=True)
    out = []
    for by_step in (True, False):
        s = _solver(dims, dtype, top, low)
        src = _wave(dims, 1.5, **kw)
        for k in steps:
            s.emsolve(k, source=src, callback=(lambda *_: None) if by_step else None)
        out.append(_state(s) + [s.nstep])
    assert out[0][0].any() and out[0][3] == out[1][3] == sum(steps)
    for name, r, g in zip("EHJ", *out):
        assert np.array_equal(r, g), f"{name} differs ({np.count_nonzero(r != g)} values)"


def test_other_runs_step_by_step():
    import wakis_amd as wa

    class Half(wa.PlaneWave):
        def update(self, solver, t):
            super().update(solver, 0.5 * t)

    dims = (12, 9, 44)
    s = _solver(dims, np.float32, "pml", "pec")
    kw = dict(zs=4, f=9 * c_light / (dims[2] * 0.8e-3), nodes=2)
    assert s._emsolve_source_steps(20, Half(**kw), 0) == 0
    assert s._emsolve_source_steps(20, wa.Dipole(), 0) == 0
    assert s._emsolve_source_steps(20, None, 0) == 0
    assert s.nstep == 0
    # a set-up whose wrap terms are dead keeps the fused path's single steps
    import wakis_amd as w
    x = np.linspace(0, 8e-3, 11)
    g = w.GridFIT3D(x=x, y=x, z=x, verbose=0)
    d = w.SolverFIT3D(g, bc_low=["pec"] * 3, bc_high=["pec"] * 3, bg=[1.0, 1.0], verbose=0)
    if d._wraps_dead():
        assert d._emsolve_source_steps(20, wa.PlaneWave(**kw), 0) == 0
