"""GPU: weight codes of the two-step kernel (wf_weight_rows, wf_weight_codes).

The table's row of every cell holds the products that the folded coefficient
arrays and the metric vectors give in FP32, value for value; pairs of steps on
weight codes leave E, H, J and the captured Ez bitwise as single steps do. Grids
whose spacing is not uniform, or with more than 255 distinct rows, have none.
"""

import numpy as np
import pytest
import torch

from tests.test_gpu_two_step import _beam_setup, _cavity_solver, _pillbox_solver

pytestmark = pytest.mark.gpu

DIMS = [(40, 13, 40), (41, 24, 33), (64, 64, 24), (256, 9, 30), (300, 40, 30)]


def _with_codes(s):
    assert s._material_table() and s._weight_table()
    return s


def _insert_solver(dims, two_step, kz=0, dtype=np.float32, bc=("pec", "pec", "pec"), x=None,
                   mats=None):
    """A dielectric block in a box that it touches: material up to the faces."""
    import wakis_amd as wa
    x = np.linspace(-5e-3, 5e-3, dims[0] + 1) if x is None else x
    y, z = (np.linspace(-5e-3, 5e-3, n + 1) for n in dims[1:])
    rng = np.random.default_rng(4)
    mats = mats or [[3.0, 1.0], [2.0, 1.5]]
    which = rng.integers(0, len(mats) + 1, dims)
    grid = wa.GridFIT3D(x=x, y=y, z=z, verbose=0,
                        stl_solids={f"m{i}": which == i for i in range(len(mats))},
                        stl_materials={f"m{i}": m for i, m in enumerate(mats)})
    s = wa.SolverFIT3D(grid, bc_low=list(bc), bc_high=list(bc), use_stl=True, bg=[1.0, 1.0],
                       dtype=dtype, verbose=0)
    s.fused_two_step, s.fused_kz = two_step, kz
    return s


@pytest.mark.parametrize("make", [_cavity_solver, _pillbox_solver, _insert_solver])
@pytest.mark.parametrize("dims", DIMS)
def test_rows_hold_the_folded_products(make, dims):
    print("weight rows", make.__name__, dims, flush=True)
    s = _with_codes(make(dims, 1))
    Nx, Ny, Nz = dims
    tab, code = s._wtab.cpu().numpy(), s._wcode.cpu().numpy().astype(int)
    assert code.min() >= 1 and code.max() < len(tab) and not tab[0].any()
    row = tab[code].reshape(Nz, Ny, Nx, -1)
    f = lambda t: t.cpu().numpy().reshape(3, Nz, Ny, Nx)
    a, b, ie, sg = f(s._a), f(s._b), f(s.ieps.array), f(s.sigma.array)
    sh = [(1, 1, Nx), (1, Ny, 1), (Nz, 1, 1)]
    L = [np.asarray(v, dtype=np.float32).reshape(h)
         for v, h in zip((s.grid.dx, s.grid.dy, s.grid.dz), sh)]
    tL = [np.asarray(v, dtype=np.float32).reshape(h) for v, h in zip(s._tL1, sh)]
    dt = np.float32(s.dt)
    for c, (u, w) in enumerate(((1, 2), (0, 2), (0, 1))):
        for q, d in enumerate((u, w)):
            assert np.array_equal(row[..., 2 * c + q], dt * (a[c] * L[d])), (c, q)
            assert np.array_equal(row[..., 6 + 2 * c + q], b[c] * tL[d]), (c, q)
        assert np.array_equal(row[..., 12 + c], ie[c])
        assert np.array_equal(row[..., 15 + c], sg[c])


@pytest.mark.parametrize("make", [_cavity_solver, _pillbox_solver])
@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("chunks,kz", [((9, 4), 0), ((7,), 5)])
def test_pairs_equal_single_steps(make, dims, chunks, kz):
    print("weight codes", make.__name__, dims, chunks, kz, flush=True)
    out = []
    for two_step in (0, 1):
        s = make(dims, two_step, kz)
        if two_step:
            _with_codes(s)
        args, cap = _beam_setup(s, sum(chunks))
        n0 = 0
        for k in chunks:
            a = args(n0, k)
            s._run(a)
            assert bool(a.wcode) == bool(two_step) and s.last_pairs == bool(two_step)
            n0 += k
        out.append([s.E.to_numpy(), s.H.to_numpy(), s.J.to_numpy(), cap.cpu().numpy()])
    assert out[0][0].any() and out[0][3].any()
    for name, r, g in zip(("E", "H", "J", "capture"), *out):
        assert np.array_equal(g, r), f"{name} differs ({np.count_nonzero(g != r)} values)"


def test_grids_without_weight_codes():
    x = np.linspace(-5e-3, 5e-3, 21) ** 3 / 25e-6
    x = x + np.linspace(-5e-3, 5e-3, 21)
    s = _insert_solver((20, 12, 14), 1, x=x)
    assert s._material_table() and not s._weight_table() and s._wcode is None
    many = _insert_solver((20, 12, 14), 1, mats=[[1.0 + 0.1 * i, 1.0] for i in range(200)])
    assert many._material_table() and not many._weight_table()  # 201 inside alone, more at the faces
    s = _insert_solver((20, 12, 14), 1)
    assert s._material_table() and s._weight_table()
    s.ieps[3:5, 3:5, 3:5, "x"] = s.ieps[3:5, 3:5, 3:5, "x"] * 0.5  # new materials, new rows
    s.update_tensors()
    before = s._wtab
    assert s._material_table() and s._weight_table() and s._wtab is not before
