"""GPU: batches that take two steps per launch (k_fused4_t2_batch).

Grids of uneven sizes and step counts whose rows are or are no whole number of
lanes, in one run and in runs of odd lengths: fields, J and wake potentials
bitwise those of each grid's own run with one step per launch. The last step of
every grid is single, so energy() works afterwards.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(dims, dtype, conductive, eps_r):
    import wakis_amd as wa
    x, y, z = (np.linspace(-0.5e-3 * n, 0.5e-3 * n, n + 1) for n in dims)
    c = [0.5 * (v[1:] + v[:-1]) for v in (x, y, z)]
    X, Y, Z = c[0][:, None, None], c[1][None, :, None], c[2][None, None, :]
    vac = (np.abs(X) < 0.4e-3 * dims[0]) & (np.abs(Y) < 0.4e-3 * dims[1]) & (
        np.abs(Z) < 0.3e-3 * dims[2]) | (X ** 2 + Y ** 2 < (3e-3) ** 2)
    ins = (np.abs(X) < 0.3e-3 * dims[0]) & (Y > 0.2e-3 * dims[1]) & (Y < 0.35e-3 * dims[1]) & (
        np.abs(Z) < 0.1e-3 * dims[2])
    mat = [eps_r, 1.0, 3.0] if conductive else [eps_r, 1.0]
    grid = wa.GridFIT3D(x=x, y=y, z=z, stl_solids={"vac": vac, "ins": ins},
                        stl_materials={"vac": "vacuum", "ins": mat}, verbose=0)
    wake = wa.WakeSolver(q=1e-9, sigmaz=3e-3, beta=1.0, skip_cells=2, save=False, verbose=0)
    return wa.SolverFIT3D(grid, wake=wake, bc_low=["pec", "pec", "abc"],
                          bc_high=["pec", "pec", "abc"], use_stl=True, bg="pec", dtype=dtype,
                          verbose=0, use_sibc=False)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("conductive", [False, True])
@pytest.mark.parametrize("sizes", [[(24, 20, 28), (40, 24, 36), (32, 44, 24)],
                                   [(23, 20, 28), (40, 25, 31), (37, 30, 26)],
                                   [(272, 9, 24), (20, 20, 20)]])
def test_pairs_match_single_grid_runs(dtype, conductive, sizes):
    from wakis_amd import batch
    print("batch pairs", np.dtype(dtype).name, conductive, sizes, flush=True)
    make = lambda: [_solver(d, dtype, conductive, 2.0 + i) for i, d in enumerate(sizes)]
    singles, batched = make(), make()
    wl = [4e-3 + 0.7e-3 * i for i in range(len(sizes))]
    for s, w in zip(singles, wl):
        s.fused_two_step = 0
        s.wakesolve(wakelength=w)
    info = batch.wakesolve_batch(batched, wl)
    assert info["tuning"] == [] and len({s.Nt for s in singles}) > 1
    for a, b in zip(singles, batched):
        for name in ("E", "H", "J"):
            assert np.array_equal(getattr(a, name).to_numpy(), getattr(b, name).to_numpy()), name
        assert np.any(b.E.to_numpy() != 0)
        assert np.array_equal(a.wake.WP_3d, b.wake.WP_3d)
        assert a.energy() == b.energy()


@pytest.mark.parametrize("chunks", [(1, 2, 3, 5, 4, 9), (7, 17), (8, 16)])
def test_runs_of_any_length(chunks):
    """The fields stay where a run of one step at a time leaves them (E2/H2 after
    an odd step), for every split of 24 steps; grids of 24, 21 and 22 steps."""
    import torch
    from wakis_amd import batch
    print("batch pairs, chunks", chunks, flush=True)
    dims = [(24, 20, 28), (32, 24, 24), (28, 28, 20)]
    total = [24, 21, 22]
    out = []
    for split in ((1,) * 24, chunks):
        sv = [_solver(d, np.float32, False, 3.0) for d in dims]
        ctxs, args = [], []
        for s, nt in zip(sv, total):
            ctx = s._wake_setup(6e-3, "both")
            a = s._wake_args(ctx, 0, nt)
            assert s._prepare_fused(a)
            a.two_step = 0 if len(split) == 24 else 1
            ctxs.append(ctx)
            args.append(a)
        b = batch._Batch(sv, args, 0, 0)
        n = 0
        states = {}
        for k in split:
            b.run(n, k, False)
            n += k
            torch.cuda.synchronize()
            states[n] = [((s._E2 if min(n, nt) % 2 else s.E.array).clone(),
                          (s._H2 if min(n, nt) % 2 else s.H.array).clone())
                         for s, nt in zip(sv, total)]
        b.close()
        out.append((states, [c["cap"].clone() for c in ctxs]))
    (ref, rcap), (got, gcap) = out
    for n in got:
        for (e0, h0), (e1, h1) in zip(ref[n], got[n]):
            assert torch.equal(e0, e1) and torch.equal(h0, h1), n
    assert all(torch.equal(a, b) for a, b in zip(rcap, gcap))
    assert all(bool((c != 0).any()) for c in gcap)
