"""GPU: who fills the region trajectory of a run on escape codes, the step kernel
(small grids) or a gather after each step (large ones, box runs, kernels that
the extra registers would hold to fewer workgroups per CU).

Either way every slot equals the gather (wf_trajectory_gather) of the fields
after the same step run alone, also where a box launches none of the block's
tiles and the fields there are what the spare buffers held.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

REG = ((3, 11), (1, 9), (5, 12))


def _block_solver(dims, dtype, cond):
    import wakis_amd as wa
    from wakis_amd.adjoint import WakeAdjoint
    x, y, z = (np.linspace(-0.5e-3 * n, 0.5e-3 * n, n + 1) for n in dims)
    blk = np.zeros(dims, dtype=bool)
    blk[tuple(slice(*r) for r in REG)] = True
    vac = np.zeros(dims, dtype=bool)
    vac[1:-1, 1:-1] = True
    grid = wa.GridFIT3D(x=x, y=y, z=z, stl_solids={"vac": vac, "blk": blk}, verbose=0,
                        stl_materials={"vac": "vacuum",
                                       "blk": [2.0, 1.0, 1.0] if cond else [2.0, 1.0]})
    wake = wa.WakeSolver(q=1e-9, sigmaz=3e-3, beta=1.0, skip_cells=2, save=False, verbose=0)
    s = wa.SolverFIT3D(grid, wake=wake, bc_low=["pec", "pec", "abc"],
                       bc_high=["pec", "pec", "abc"], use_stl=True, bg="pec", dtype=dtype,
                       verbose=0, use_sibc=False)
    s.code_escape_max = 0.2
    adj = WakeAdjoint(s, REG, 2e-3, mode="trajectory")
    rng = np.random.default_rng(3)
    sh = adj.shape
    adj._set_params(rng.uniform(1, 10, sh), rng.uniform(0, 2, sh) if cond else None)
    return s, adj


def _slots(adj, n):
    dt, dev = adj.s.E.array.dtype, adj.s.device
    return tuple(torch.full((n, 3 * m), 7.0, dtype=dt, device=dev) for m in (adj._nE, adj._nH))


def _with_slots(args, adj, tE, tH):
    from wakis_amd import _lib
    args.traj_E, args.traj_H = _lib.ptr(tE), _lib.ptr(tH)
    args.traj_lo[:], args.traj_hi[:] = tuple(a for a, _ in REG), tuple(b for _, b in REG)
    args.traj_slots, args.traj_slot0 = tE.shape[0], 0
    return args


def _gather(adj):
    from wakis_amd import _lib
    s = adj.s
    tE, tH = _slots(adj, 1)
    lo, hi = adj._lohi()
    _lib.check(_lib.lib().wf_trajectory_gather(
        s._handle, _lib.ptr(s.E.array), _lib.ptr(s.H.array), _lib.ptr(tE), _lib.ptr(tH), lo, hi,
        1, 0, _lib.stream_ptr()), "wf_trajectory_gather")
    return tE[0], tH[0]


# in the step up to 2^19 cells: (64, 64, 128) is the last such size; FP64 rows of
# two cells a lane with conduction lose a workgroup per CU and are gathered
@pytest.mark.parametrize("dims", [(24, 20, 26), (72, 14, 22), (64, 64, 128), (64, 64, 129)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("cond", [True, False])
def test_slots_equal_the_gather(dims, dtype, cond):
    print("trajectory rule", dims, np.dtype(dtype).name, cond, flush=True)
    s, adj = _block_solver(dims, dtype, cond)
    n = 9
    ctx = s._wake_setup(adj.wakelength, "both")
    tE, tH = _slots(adj, n + 1)
    s._run(_with_slots(s._wake_args(ctx, 0, n), adj, tE, tH))
    assert s._code_escape and s.last_path == "fused"
    s.reset_fields()
    ctx = s._wake_setup(adj.wakelength, "both")
    for i in range(n):
        s._run(s._wake_args(ctx, i, 1))
        e, h = _gather(adj)
        assert torch.equal(e, tE[i + 1]) and torch.equal(h, tH[i + 1]), i
    assert bool((tE[1:] != 7).all()) and bool((tH[1:] != 7).all())


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_box_that_misses_part_of_the_block(dtype):
    print("trajectory of a box", np.dtype(dtype).name, flush=True)
    s, adj = _block_solver((24, 20, 26), dtype, True)
    ctx = s._wake_setup(adj.wakelength, "both")
    s._run(s._wake_args(ctx, 0, 20))
    for spare in (s._E2, s._H2):
        spare.fill_(3.0)
    tE, tH = _slots(adj, 2)
    args = _with_slots(s._wake_args(ctx, 20, 1), adj, tE, tH)
    args.box_lo[:], args.box_hi[:] = (4, 2, 5), (6, 3, 6)
    s._run(args)
    e, h = _gather(adj)  # the step's output buffers: the box's tiles, 3.0 elsewhere
    assert bool((e == 3).any()) and bool((e != 3).any())
    assert torch.equal(e, tE[1]) and torch.equal(h, tH[1])
