"""GPU: a field monitor on runs of two steps per launch.

The E of 2, 4 or 8 steps is accumulated in one pass over the accumulators
(``wf_step_args.mon_work``): accumulators, fields and wake bitwise those of one
step per launch with one pass per step, for every size of the scratch, calls
that end anywhere in a pass, rows that are no whole number of lanes, FP32 and
FP64, with and without conduction, and any number of frequencies.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(dims, dtype, conductive, slots, chunk, freqs):
    import wakis_amd as wa
    from wakis_amd import FieldMonitor
    x, y, z = (np.linspace(-0.5e-3 * n, 0.5e-3 * n, n + 1) for n in dims)
    c = [0.5 * (v[1:] + v[:-1]) for v in (x, y, z)]
    vac = ((np.abs(c[0]) < 0.4e-3 * dims[0])[:, None, None]
           & (np.abs(c[1]) < 0.4e-3 * dims[1])[None, :, None] & np.ones(dims, dtype=bool))
    ins = vac & (c[1] > 0.2e-3 * dims[1])[None, :, None]
    grid = wa.GridFIT3D(x=x, y=y, z=z, stl_solids={"vac": vac, "ins": ins},
                        stl_materials={"vac": "vacuum",
                                       "ins": [3.0, 1.0, 2.0] if conductive else [3.0, 1.0]},
                        verbose=0)
    wake = wa.WakeSolver(q=1e-9, sigmaz=3e-3, beta=1.0, skip_cells=2, save=False, verbose=0)
    s = wa.SolverFIT3D(grid, wake=wake, bc_low=["pec", "pec", "abc"],
                       bc_high=["pec", "pec", "abc"], use_stl=True, bg="pec", dtype=dtype,
                       verbose=0, use_sibc=False)
    if slots is None:
        s.fused_two_step = 0
    else:
        s._monitor_work = lambda: torch.full((slots, 3 * s.N), float("nan"),
                                             dtype=s.E.array.dtype, device=s.device)
    m = FieldMonitor(freqs)
    s.wakesolve(wakelength=3e-3, use_field_monitor=True, field_monitor=m, chunk=chunk)
    return s, m


@pytest.mark.parametrize("dims,chunk,freqs", [((24, 20, 24), None, [1e9, 2.5e9]),
                                              ((23, 17, 22), 19, [1e9]),
                                              ((20, 33, 21), 6, [0.5e9, 1e9, 2e9, 4e9, 5e9])])
@pytest.mark.parametrize("slots", [1, 3, 7, 12])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("conductive", [False, True])
def test_passes_over_several_steps(dims, chunk, freqs, slots, dtype, conductive):
    print("monitor pairs", dims, chunk, slots, np.dtype(dtype).name, conductive, flush=True)
    s1, m1 = _run(dims, dtype, conductive, None, chunk, freqs)
    s2, m2 = _run(dims, dtype, conductive, slots, chunk, freqs)
    assert not s1.last_pairs and s1.Nt == s2.Nt and m1.time_index == m2.time_index
    assert chunk is not None or s2.last_pairs
    for name in ("E", "H", "J"):
        assert torch.equal(getattr(s1, name).array, getattr(s2, name).array), name
    for c in ("Ex", "Ey", "Ez"):
        a, b = m1.get_components()[c], m2.get_components()[c]
        assert torch.equal(a, b) and bool((b != 0).any()), c
    assert np.array_equal(s1.wake.WP_3d, s2.wake.WP_3d)
    assert s1.energy() == s2.energy()
