"""GPU: a monitored wakesolve holds scratch for the E of several steps only where
its calls take two steps per launch, and no more of it than a call can use."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(**attrs):
    import wakis_amd as wa
    x = np.linspace(-6e-3, 6e-3, 13)
    z = np.linspace(-10e-3, 10e-3, 21)
    vac = np.zeros((12, 12, 20), dtype=bool)
    vac[1:-1, 1:-1] = True
    grid = wa.GridFIT3D(x=x, y=x, z=z, stl_solids={"v": vac}, stl_materials={"v": "vacuum"},
                        verbose=0)
    wake = wa.WakeSolver(q=1e-9, sigmaz=3e-3, beta=1.0, skip_cells=2, save=False, verbose=0)
    s = wa.SolverFIT3D(grid, wake=wake, bc_low=["pec", "pec", "abc"],
                       bc_high=["pec", "pec", "abc"], use_stl=True, bg="pec", dtype=np.float32,
                       verbose=0)
    for k, v in attrs.items():
        setattr(s, k, v)
    return s


@pytest.mark.parametrize("attrs,kw,slots", [
    ({}, {}, 7), ({}, {"chunk": 9}, 7), ({}, {"chunk": 8}, 5), ({}, {"chunk": 6}, 3),
    ({}, {"chunk": 3}, 1), ({}, {"chunk": 2}, None),
    ({}, {"callback": lambda s, t: None}, None),
    ({"fused_two_step": 0}, {}, None), ({"path": "general"}, {}, None),
    ({"use_material_code": False}, {}, None)])
def test_scratch_is_what_the_calls_use(attrs, kw, slots):
    from wakis_amd import FieldMonitor
    print("monitor scratch", attrs, list(kw), slots, flush=True)
    got, ref = [], None
    for s, run in ((_solver(fused_two_step=0), {}), (_solver(**attrs), kw)):
        make = s._monitor_work

        def counted():
            got.append(make())
            return got[-1]
        s._monitor_work = counted
        m = FieldMonitor([1e9, 4e9])
        s.wakesolve(wakelength=2e-3, use_field_monitor=True, field_monitor=m, **run)
        acc = m.get_components()
        if ref is None:
            assert got == []
            ref = acc
    assert [w.shape[0] for w in got] == ([] if slots is None else [slots])
    for c in ("Ex", "Ey", "Ez"):
        assert bool((acc[c] == ref[c]).all()) and bool((acc[c] != 0).any()), c
