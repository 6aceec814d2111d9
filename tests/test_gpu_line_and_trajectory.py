"""GPU: the beam line written from kernel arguments (wf_write_line) and the
region trajectory filled by the escape-code step kernels themselves.

The line equals the values rounded to the field dtype, for lengths around the
chunk of one launch, and nothing else changes. The trajectory equals, slot by
slot, the gather (wf_trajectory_gather) of the fields after each single step.
"""

import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,nz", [(np.float32, 20), (np.float32, 768), (np.float32, 769),
                                      (np.float64, 384), (np.float64, 385), (np.float64, 1000)])
def test_beam_line_values(dtype, nz):
    import wakis_amd as wa
    print("beam line", np.dtype(dtype).name, nz, flush=True)
    x = np.linspace(0, 4e-3, 5)
    z = np.linspace(0, 1e-3 * nz, nz + 1)
    s = wa.SolverFIT3D(wa.GridFIT3D(x=x, y=x, z=z, verbose=0), bc_low=["pec"] * 3,
                       bc_high=["pec"] * 3, bg=[1.0, 1.0], dtype=dtype, verbose=0)
    s.J.array.uniform_(-1, 1)
    want = s.J.to_numpy().reshape(3, nz, 4, 4)
    vals = np.random.default_rng(nz).standard_normal(nz) * 1e3
    v0 = s.J.version
    s._write_beam_line(2, 1, vals)
    want[2, :, 1, 2] = vals.astype(dtype)
    assert np.array_equal(s.J.to_numpy().reshape(want.shape), want)
    assert s._beam_line == (2, 1) and s.J.version == v0
    with pytest.raises(IndexError):
        s._write_beam_line(4, 1, vals)


@pytest.mark.parametrize("dims,lanes,rows", [((24, 20, 26), 0, 0), ((24, 20, 26), 4, 0),
                                             ((23, 20, 26), 1, 0), ((72, 14, 22), 4, 2)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_trajectory_of_escape_kernels(dims, lanes, rows, dtype):
    import wakis_amd as wa
    from wakis_amd import _lib
    from wakis_amd.adjoint import WakeAdjoint
    if dtype == np.float64 and lanes == 4:
        lanes = 2
    print("trajectory", dims, lanes, rows, np.dtype(dtype).name, flush=True)
    x, y, z = (np.linspace(-0.5e-3 * n, 0.5e-3 * n, n + 1) for n in dims)
    reg = ((3, 11), (1, 8), (5, 12))
    blk = np.zeros(dims, dtype=bool)
    blk[tuple(slice(*r) for r in reg)] = True
    vac = np.zeros(dims, dtype=bool)
    vac[1:-1, 1:-1] = True
    grid = wa.GridFIT3D(x=x, y=y, z=z, stl_solids={"vac": vac, "blk": blk},
                        stl_materials={"vac": "vacuum", "blk": [2.0, 1.0, 1.0]}, verbose=0)
    wake = wa.WakeSolver(q=1e-9, sigmaz=3e-3, beta=1.0, skip_cells=2, save=False, verbose=0)
    s = wa.SolverFIT3D(grid, wake=wake, bc_low=["pec", "pec", "abc"],
                       bc_high=["pec", "pec", "abc"], use_stl=True, bg="pec", dtype=dtype,
                       verbose=0, use_sibc=False)
    s.code_escape_max = 0.2
    s.fused_cells_per_lane, s.fused_full_rows = lanes, rows
    rng = np.random.default_rng(3)
    sh = tuple(b - a for a, b in reg)
    adj = WakeAdjoint(s, reg, 2e-3, mode="trajectory")
    adj.forward(rng.uniform(1, 10, sh), rng.uniform(0, 2, sh))
    assert s._code_escape and s.last_path == "fused"
    tE, tH = adj._fwd["traj"]
    Nt = min(adj._fwd["Nt"], 60)
    ctx = s._wake_setup(adj.wakelength, "both")
    s.reset_fields()
    s._set_ghosts_to_0()
    lo, hi = adj._lohi()
    oE, oH = torch.zeros_like(tE[:1]), torch.zeros_like(tH[:1])
    ctx = s._wake_setup(adj.wakelength, "both")
    for n in range(Nt):
        s._run(s._wake_args(ctx, n, 1))
        _lib.check(_lib.lib().wf_trajectory_gather(
            s._handle, _lib.ptr(s.E.array), _lib.ptr(s.H.array), _lib.ptr(oE), _lib.ptr(oH),
            lo, hi, 1, 0, _lib.stream_ptr()), "wf_trajectory_gather")
        assert torch.equal(oE[0], tE[n + 1]) and torch.equal(oH[0], tH[n + 1]), n
    assert bool((oE != 0).any()) and bool((oH != 0).any())
