"""The work a user of wakis_amd has it do, as cases that can be timed and checked.

``listed()`` names the cases, ``draw(rng)`` gives further ones from the same
ranges, ``prepare(case, seed)`` makes what a program holds before the call,
``run(state)`` is one pass through the public entry points, ``work(case)`` the
bytes and operations a pass cannot do without, and ``exact(case, seed)`` the
same outputs from plain numpy and torch in 64 bits.

Kinds of case:

* ``wake``    ``SolverFIT3D.wakesolve`` from zero fields: step loop, Ez capture,
              wake potentials, impedances (optionally with a ``FieldMonitor``).
* ``loop``    the user loop of the reference's examples: ``Beam.update`` and
              ``one_step`` per step.
* ``emsolve`` ``emsolve`` with a plane wave, periodic in x and y, PML or ABC in z.
* ``batch``   ``wakesolve_batch`` over many small cavities.
* ``adjoint`` ``WakeAdjoint.forward`` and ``backward`` (loss and gradients).
* ``post``    ``WakeSolver.solve`` again on the samples of a finished run.
"""

import math
import random

import numpy as np
import torch

C = 299792458.0
MU0 = 1.25663706127e-06
EPS0 = 8.8541878188e-12
EXACT_MAX_CELL_STEPS = 3.0e10  # above this the 64-bit run takes too long


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the step loop written by hand on a small grid: latency of one call
        dict(name="loop-40x40x64-f32", kind="loop", nx=40, ny=40, nz=64, cell=1.2e-3, dz=1.2e-3,
             dtype="float32", steps=200, sigmaz=6e-3),
        # the 48x48x128 cavity with pipe, 0.5 m wake, default precision: an
        # everyday small run, 2,062 steps of a few microseconds of work each
        dict(name="wake-48x48x128-f64", kind="wake", shape="cavity", nx=48, ny=48, nz=128,
             cell=1.25e-3, dz=1.25e-3, dtype="float64", sigmaz=10e-3, wl=0.5, plane="both",
             nfreq=0),
        # a ragged grid, as a cell size picked by hand gives it; longitudinal only
        dict(name="wake-91x75x161-f32", kind="wake", shape="cavity", nx=91, ny=75, nz=161,
             cell=0.7e-3, dz=0.8e-3, dtype="float32", sigmaz=8e-3, wl=0.06,
             plane="longitudinal", nfreq=0),
        # an ordinary run in the default precision
        dict(name="wake-160x160x200-f64", kind="wake", shape="cavity", nx=160, ny=160, nz=200,
             cell=0.4e-3, dz=0.5e-3, dtype="float64", sigmaz=6e-3, wl=0.02, plane="both",
             nfreq=0),
        # the throughput workload: 256x256x512 cells, FP32
        dict(name="wake-256x256x512-f32", kind="wake", shape="cavity", nx=256, ny=256, nz=512,
             cell=60e-3 / 256, dz=160e-3 / 512, dtype="float32", sigmaz=10e-3, wl=0.02,
             plane="both", nfreq=0, insert=False),
        # a wide structure: rows of more than 256 cells
        dict(name="wake-300x220x180-f32", kind="wake", shape="cavity", nx=300, ny=220, nz=180,
             cell=0.4e-3, dz=0.4e-3, dtype="float32", sigmaz=4e-3, wl=0.01, plane="both",
             nfreq=0),
        # the lossy pillbox with PML (conduction everywhere)
        dict(name="wake-pillbox-200x200x400-f32", kind="wake", shape="pillbox", nx=200, ny=200,
             nz=400, cell=0.45e-3, dz=0.45e-3, dtype="float32", sigmaz=4e-3, wl=0.01,
             plane="both", nfreq=0),
        # field maps at two frequencies accumulated during a run
        dict(name="wake-monitor-96x96x160-f32", kind="wake", shape="cavity", nx=96, ny=96,
             nz=160, cell=0.7e-3, dz=0.8e-3, dtype="float32", sigmaz=8e-3, wl=0.03,
             plane="both", nfreq=2),
        # plane wave into a PML, periodic in x and y, source written every step
        dict(name="emsolve-64x64x60-f32", kind="emsolve", nx=64, ny=64, nz=60, cell=0.8e-3,
             dz=0.8e-3, dtype="float32", steps=240, top="pml"),
        # a parameter sweep over many small cavities
        dict(name="batch-24-f32", kind="batch", n=24, dims_lo=28, dims_hi=80, mix=5,
             dtype="float32", steps=600),
        # gradient of the wake figure of merit with respect to a block's cells
        dict(name="adjoint-64x64x96-f32", kind="adjoint", nx=64, ny=64, nz=96, cell=0.9e-3,
             dz=1.0e-3, block=16, dtype="float32", sigmaz=8e-3, wl=0.03),
        # the post-processing alone, evaluated again on a finished long run
        dict(name="post-20x20x300-f64", kind="post", nx=20, ny=20, nz=300, cell=1e-3, dz=1e-3,
             dtype="float64", sigmaz=8e-3, steps=8000),
    ]


def _lu(rng, lo, hi):
    """An integer, uniform in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loop", "wake", "wake", "wake", "wake", "wake-small", "monitor",
                       "emsolve", "batch", "adjoint", "post"])
    dtype = rng.choice(["float32", "float32", "float64"])
    cell = rng.uniform(0.35e-3, 1.2e-3)
    dz = cell * rng.uniform(1.0, 1.3)
    if kind == "loop":
        return dict(kind="loop", nx=_lu(rng, 20, 160), ny=_lu(rng, 20, 160),
                    nz=_lu(rng, 24, 200), cell=cell, dz=dz, dtype=dtype,
                    steps=_lu(rng, 50, 300), sigmaz=cell * rng.uniform(4, 10))
    if kind in ("wake", "wake-small", "monitor"):
        small = kind != "wake"
        shape = rng.choice(["cavity", "cavity", "pillbox"])
        if shape == "pillbox":  # the PML's time constant: cells below 0.8 mm
            cell = rng.uniform(0.3e-3, 0.6e-3)
            dz = cell
        nx, ny = _lu(rng, 30, 110 if small else 340), _lu(rng, 30, 110 if small else 300)
        nz = _lu(rng, 48, 200 if small else 420)
        sigmaz = cell * rng.uniform(8, 14)
        return dict(kind="wake", shape=shape, nx=nx, ny=ny, nz=nz, cell=cell, dz=dz,
                    dtype=dtype, sigmaz=sigmaz, wl=cell * rng.uniform(20, 120),
                    plane=rng.choice(["both", "both", "longitudinal"]),
                    nfreq=rng.choice([1, 2, 3]) if kind == "monitor" else 0)
    if kind == "emsolve":
        return dict(kind="emsolve", nx=_lu(rng, 12, 128), ny=_lu(rng, 12, 128),
                    nz=_lu(rng, 40, 200), cell=0.8e-3, dz=0.8e-3, dtype=dtype,
                    steps=_lu(rng, 60, 300), top=rng.choice(["pml", "abc"]))
    if kind == "batch":
        return dict(kind="batch", n=rng.randint(4, 24), dims_lo=24, dims_hi=_lu(rng, 40, 88),
                    mix=rng.randint(0, 999), dtype=dtype, steps=_lu(rng, 300, 900))
    if kind == "adjoint":
        return dict(kind="adjoint", nx=_lu(rng, 40, 110), ny=_lu(rng, 40, 110),
                    nz=_lu(rng, 56, 140), cell=cell, dz=dz, block=rng.randint(6, 20),
                    dtype=dtype, sigmaz=cell * rng.uniform(8, 10),
                    wl=cell * rng.uniform(20, 120))
    return dict(kind="post", nx=_lu(rng, 16, 32), ny=_lu(rng, 16, 32), nz=_lu(rng, 60, 400),
                cell=1e-3, dz=1e-3, dtype=dtype, sigmaz=8e-3, steps=_lu(rng, 2500, 9000))


# ------------------------------------------------------------ problem set-up
def _axes(nx, ny, nz, cell, dz):
    return (np.linspace(-nx * cell / 2, nx * cell / 2, nx + 1),
            np.linspace(-ny * cell / 2, ny * cell / 2, ny + 1),
            np.linspace(-nz * dz / 2, nz * dz / 2, nz + 1))


def _centres(v):
    return v[:-1] + np.diff(v) / 2


def _grow(m):
    g = m.copy()
    for ax in range(3):
        a, b = np.moveaxis(g, ax, 0), np.moveaxis(m, ax, 0)
        a[1:] |= b[:-1]
        a[:-1] |= b[1:]
    return g


def _structure(case, seed):
    """The set-up of a beam-driven case: axes, solids (cell masks and
    materials), boundaries and beam; the seed moves the beam and the test line
    by up to a cell and sets the insert's permittivity and the charge."""
    rng = np.random.default_rng(1000 + seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cell, dz = case["cell"], case["dz"]
    x, y, z = _axes(nx, ny, nz, cell, dz)
    X, Y, Z = (_centres(x)[:, None, None], _centres(y)[None, :, None],
               _centres(z)[None, None, :])
    hx, hy, hz = -x[0], -y[0], -z[0]
    rp = 0.25 * min(hx, hy)
    eps_r = float(rng.uniform(2.0, 6.0))
    shape = case.get("shape", "cavity")
    if shape == "pillbox":
        R2 = X ** 2 + Y ** 2
        vac = ((R2 < (0.85 * min(hx, hy)) ** 2) & (np.abs(Z) < 0.4 * hz)) | (R2 < rp ** 2)
        wall = _grow(_grow(vac)) & ~vac
        solids = [("vacuum", vac, [1.0, 1.0]), ("wall", wall, [eps_r, 1.0, 2.0])]
        bc = ["pec", "pec", "pml"]
    else:
        vac = (((np.abs(X) < 0.83 * hx) & (np.abs(Y) < 0.83 * hy) & (np.abs(Z) < 0.35 * hz))
               | (X ** 2 + Y ** 2 < rp ** 2))
        ins = ((np.abs(X) > 0.5 * hx) & (np.abs(X) < 0.8 * hx) & (np.abs(Y) < 0.5 * hy)
               & (np.abs(Z) < 0.2 * hz))
        solids = [("vacuum", vac, [1.0, 1.0]), ("insert", ins, [eps_r, 1.0])]
        if not case.get("insert", True):  # the empty cavity, its walls moved by the seed
            solids = [("vacuum", vac & (np.abs(X) < (0.8 + 0.005 * eps_r) * hx), [1.0, 1.0])]
        bc = ["pec", "pec", "abc"]
    off = rng.integers(-1, 2, 4) * cell
    return dict(x=x, y=y, z=z, solids=solids, bc=(bc, bc), bg="pec", dtype=case["dtype"],
                q=float(rng.uniform(0.5e-9, 2e-9)), sigmaz=case["sigmaz"],
                xs=float(off[0]), ys=float(off[1]), xt=float(off[2]), yt=float(off[3]),
                skip=0 if case.get("plane") == "longitudinal" else max(1, nz // 20))


def _dt(p):
    d = [np.min(np.diff(v)) for v in (p["x"], p["y"], p["z"])]
    return np.dtype(p["dtype"]).type(0.5 / (C * np.sqrt(1 / d[0] ** 2 + 1 / d[1] ** 2
                                                       + 1 / d[2] ** 2)))


def _ti(p):
    return 8.548921333333334 * p["sigmaz"] / C


def _wl_for_steps(p, steps):
    """Wake length of a run of about ``steps`` steps."""
    z = _centres(p["z"])
    return float((steps + 0.5) * float(_dt(p)) * C - _ti(p) * C - (z.max() - z.min()))


def _steps_of_wl(p, wl):
    z = _centres(p["z"])
    return int((wl + _ti(p) * C + (z.max() - z.min())) / C / _dt(p))


def _batch_structures(case, seed):
    """The cavities of a sweep: sizes from ``mix``, permittivities and charges
    from the seed."""
    mix = random.Random(case["mix"])
    out = []
    for i in range(case["n"]):
        nx, ny = (4 * (mix.randint(case["dims_lo"], case["dims_hi"]) // 4) for _ in range(2))
        nz = 4 * (mix.randint(case["dims_lo"], 2 * case["dims_hi"]) // 4)
        c = dict(nx=nx, ny=ny, nz=nz, cell=1e-3, dz=1e-3, dtype=case["dtype"], sigmaz=5e-3)
        p = _structure(c, 7919 * seed + i)
        # the sweep's steps, or as many as its longest grid needs to hold the axis
        out.append((p, max(_wl_for_steps(p, case["steps"]), 0.01)))
    return out


def _solver(p, **kw):
    import wakis_amd as wa
    grid = wa.GridFIT3D(x=p["x"], y=p["y"], z=p["z"],
                        stl_solids={k: m for k, m, _ in p["solids"]},
                        stl_materials={k: mat for k, _, mat in p["solids"]}, verbose=0)
    wake = wa.WakeSolver(q=p["q"], sigmaz=p["sigmaz"], beta=1.0, xsource=p["xs"],
                         ysource=p["ys"], xtest=p["xt"], ytest=p["yt"], skip_cells=p["skip"],
                         save=False, verbose=0)
    return wa.SolverFIT3D(grid, wake=wake, bc_low=p["bc"][0], bc_high=p["bc"][1],
                          use_stl=True, bg=p["bg"], dtype=np.dtype(p["dtype"]).type, verbose=0,
                          **kw)


def _block_region(case):
    b = case["block"]
    n = (case["nx"], case["ny"], case["nz"])
    e = [min(b, v // 3) for v in n]
    lo = [n[0] // 2 + 2 if n[0] // 2 + 2 + e[0] < n[0] else n[0] // 3,
          (n[1] - e[1]) // 2, (n[2] - e[2]) // 2]
    return tuple((a, a + m) for a, m in zip(lo, e))


def _block_values(case, seed):
    reg = _block_region(case)
    sh = tuple(b - a for a, b in reg)
    rng = np.random.default_rng(2000 + seed)
    return rng.uniform(1.0, 10.0, sh), rng.uniform(0.0, 2.0, sh)


def _adjoint_structure(case, seed):
    p = _structure(case, seed)
    ins = np.zeros((case["nx"], case["ny"], case["nz"]), dtype=bool)
    ins[tuple(slice(a, b) for a, b in _block_region(case))] = True
    p["solids"] = [p["solids"][0], ("block", ins, [2.0, 1.0, 1.0])]
    return p


def _plane_wave(case, seed):
    rng = np.random.default_rng(3000 + seed)
    length = case["nz"] * case["dz"]
    return dict(zs=5, nodes=float(rng.uniform(2.0, 7.0)), f=float(rng.uniform(8, 20)) * C / length,
                amplitude=float(rng.uniform(1.0, 10.0)), phase=float(rng.uniform(0, np.pi)))


def _em_structure(case):
    x, y, z = _axes(case["nx"], case["ny"], case["nz"], case["cell"], case["dz"])
    low = "pec" if case["top"] == "pml" else "abc"
    return dict(x=x, y=y, z=z, solids=[], bc=(["periodic", "periodic", low],
                                             ["periodic", "periodic", case["top"]]),
                bg=[1.0, 1.0], dtype=case["dtype"])


# ------------------------------------------------------------ prepare and run
def prepare(case, seed):
    import wakis_amd as wa
    kind = case["kind"]
    st = dict(kind=kind, case=case)
    if kind == "wake":
        st["solver"] = _solver(_structure(case, seed))
        st["freqs"] = [1.1e9 + 0.9e9 * i for i in range(case["nfreq"])]
    elif kind == "loop":
        p = _structure(case, seed)
        st["solver"] = _solver(p)
        st["beam"] = wa.Beam(q=p["q"], sigmaz=p["sigmaz"], xsource=p["xs"], ysource=p["ys"],
                             ti=2.0 * p["sigmaz"] / C)
    elif kind == "emsolve":
        p = _em_structure(case)
        grid = wa.GridFIT3D(x=p["x"], y=p["y"], z=p["z"], verbose=0)
        st["solver"] = wa.SolverFIT3D(grid, bc_low=p["bc"][0], bc_high=p["bc"][1], bg=p["bg"],
                                      dtype=np.dtype(p["dtype"]).type, verbose=0)
        st["source"] = wa.PlaneWave(**_plane_wave(case, seed))
    elif kind == "batch":
        ps = _batch_structures(case, seed)
        st["solvers"] = [_solver(p) for p, _ in ps]
        st["wl"] = [w for _, w in ps]
    elif kind == "adjoint":
        from wakis_amd.adjoint import WakeAdjoint
        p = _adjoint_structure(case, seed)
        s = _solver(p, use_sibc=False, tau_clamp=False)
        st["adj"] = WakeAdjoint(s, _block_region(case), case["wl"], w_loss=1.0, w_band=1e-13)
        st["eps_r"], st["sigma"] = _block_values(case, seed)
    else:  # post: a finished run
        p = _structure(case, seed)
        s = _solver(p)
        s.wakesolve(_wl_for_steps(p, case["steps"]))
        st["wake"] = s.wake
    return st


def _reset(s):
    """The solver as it was before its first step."""
    s.reset_fields()
    s.step_0 = True


def _join(outs):
    """One result per quantity from many grids': the values end to end."""
    return {k: np.concatenate([np.atleast_1d(o[k]).reshape(-1) for o in outs]) for k in outs[0]}


def _wake_out(w, plane):
    out = dict(s=w.s, WP=w.WP, f=w.f, Z=w.Z, loss=w.loss_factor)
    if plane == "both":
        out.update(WP_3d=w.WP_3d, WPx=w.WPx, WPy=w.WPy, Zx=w.Zx, Zy=w.Zy)
    return out


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "wake":
        s = state["solver"]
        kw = {}
        if state["freqs"]:
            from wakis_amd.field_monitors import FieldMonitor
            kw = dict(use_field_monitor=True, field_monitor=FieldMonitor(state["freqs"]))
        _reset(s)
        s.wakesolve(case["wl"], compute_plane=case["plane"], **kw)
        out = _wake_out(s.wake, case["plane"])
        out.update(E=s.E.array, H=s.H.array)
        if state["freqs"]:
            out.update(kw["field_monitor"].get_components())
        return out
    if kind == "loop":
        s, beam = state["solver"], state["beam"]
        _reset(s)
        for n in range(case["steps"]):
            beam.update(s, n * s.dt)
            s.one_step()
        return dict(E=s.E.array, H=s.H.array)
    if kind == "emsolve":
        s = state["solver"]
        _reset(s)
        s.emsolve(case["steps"], source=state["source"])
        return dict(E=s.E.array, H=s.H.array, J=s.J.array)
    if kind == "batch":
        from wakis_amd.batch import wakesolve_batch
        sv = state["solvers"]
        for s in sv:
            _reset(s)
        wakesolve_batch(sv, state["wl"])
        return dict(_join([_wake_out(s.wake, "both") for s in sv]),
                    E=[s.E.array for s in sv], H=[s.H.array for s in sv])
    if kind == "adjoint":
        adj = state["adj"]
        L = adj.forward(state["eps_r"], state["sigma"])
        ge, gs = adj.backward()
        return dict(L=L, g_eps=ge, g_sigma=gs)
    w = state["wake"]
    w.solve(compute_plane="both")
    return _wake_out(w, "both")


def work(case):
    """A pass reads the materials once and writes the final fields (and results)
    once; every step costs 54 operations per cell (four products, three sums,
    the scaling and the update of six components), 60 with conduction."""
    it = np.dtype(case["dtype"]).itemsize

    def step_work(n, steps, cond=False):
        return dict(bytes=((9 if cond else 6) + 6) * n * it + 8 * 9 * steps,
                    flops=(60 if cond else 54) * n * steps)

    kind = case["kind"]
    if kind == "batch":
        tot = dict(bytes=0, flops=0)
        for p, wl in _batch_structures(case, 0):
            n = math.prod(len(p[a]) - 1 for a in "xyz")
            w = step_work(n, _steps_of_wl(p, wl))
            tot = {k: tot[k] + w[k] for k in tot}
        return tot
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "wake":
        p = _structure_axes(case)
        steps = _steps_of_wl(p, case["wl"])
        w = step_work(n, steps, case["shape"] == "pillbox")
        w["bytes"] += 48 * n * case["nfreq"]
        w["flops"] += 12 * n * case["nfreq"] * steps
        return w
    if kind == "post":
        p = _structure_axes(case)
        steps = case["steps"]
        lines, bins = 9, 1001
        return dict(bytes=lines * steps * case["nz"] * it,
                    flops=2 * lines * steps * case["nz"] + 5 * 4 * bins * steps)
    if kind == "adjoint":  # the step and its transpose, conduction in both
        p = _structure_axes(case)
        w = step_work(n, _steps_of_wl(p, case["wl"]), True)
        return dict(bytes=w["bytes"], flops=2 * w["flops"])
    return step_work(n, case["steps"], kind == "emsolve" and case["top"] == "pml")


def _structure_axes(case):
    x, y, z = _axes(case["nx"], case["ny"], case["nz"], case["cell"], case["dz"])
    return dict(x=x, y=y, z=z, dtype=case["dtype"], sigmaz=case["sigmaz"])


# ------------------------------------------------------- the same in 64 bits
class _Sim:
    """The FIT leapfrog in 64 bits on flat component arrays: H -= dt a (C L E),
    E += dt (b C^T tL H - J/eps), J = sigma E, differences over the flat index
    (x fastest) cut at the ends, PEC faces as zero columns and rows."""

    def __init__(self, p, n_pml=10):
        self.dev = torch.device("cuda")
        self.x, self.y, self.z = (_centres(p[a]) for a in "xyz")
        nx, ny, nz = self.n = tuple(len(p[a]) - 1 for a in "xyz")
        self.N, self.sy, self.sz = nx * ny * nz, nx, nx * ny
        self.dt = float(_dt(p))
        lo, hi = ([b.lower() for b in side] for side in p["bc"])
        L = [np.diff(p[a]) for a in "xyz"]
        tL = [np.append(0.5 * (v[1:] + v[:-1]), 0.0) for v in L]
        self.dx, self.dy, self.dz = L
        shp = [(1, 1, nx), (1, ny, 1), (nz, 1, 1)]
        full = lambda v, a: np.broadcast_to(v.reshape(shp[a]), (nz, ny, nx))
        edits = [a for a in range(3) if (lo[a] == hi[a] == "periodic") or hi[a] == "abc"]
        # materials
        if p["bg"] == "pec":
            ie0, im0, sg0 = 0.0, 1 / MU0, 0.0
        else:
            ie0, im0, sg0 = 1 / (p["bg"][0] * EPS0), 1 / (p["bg"][1] * MU0), 0.0
        ie, im, sg = (np.full((nz, ny, nx), v) for v in (ie0, im0, sg0))
        cond = False
        for _, m, mat in p["solids"]:
            mt = np.transpose(m, (2, 1, 0))
            ie[mt], im[mt] = 1 / (mat[0] * EPS0), 1 / (mat[1] * MU0)
            if len(mat) == 3:
                sg[mt] = mat[2]
                cond = True
        for side, b in ((0, lo), (1, hi)):
            for a in range(3):
                if b[a] != "pml":
                    continue
                cond = True
                prof = np.geomspace(10.0, 5e-3, n_pml)
                c = [nx // 2, ny // 2, nz // 2]
                c[a] = n_pml + 1 if side == 0 else self.n[a] - (n_pml + 1)
                i0, s0 = ie[c[2], c[1], c[0]], sg[c[2], c[1], c[0]]
                for m in range(n_pml):
                    sl = [slice(None)] * 3
                    sl[2 - a] = m if side == 0 else self.n[a] - 1 - m
                    ie[tuple(sl)] = i0
                    sg[tuple(sl)] = s0 + (1 if s0 < 1 else s0) * prof[m]
        t = lambda v: torch.as_tensor(np.ascontiguousarray(v), device=self.dev).reshape(-1)
        self.ie, self.sg, self.cond = t(ie), t(sg), cond
        pec = lambda b: b in ("pec", "pml", "electric")
        self.a, self.b, self.L, self.tL = [], [], [], []
        for c in range(3):
            u, w = [d for d in range(3) if d != c]
            iA = 1.0 / (full(L[u], u) * full(L[w], w))
            aux = full(tL[u], u) * full(tL[w], w)
            itA = np.divide(1.0, aux, out=np.zeros((nz, ny, nx)), where=aux != 0)
            for e in edits:
                if e != c:
                    np.moveaxis(itA, 2 - e, 0)[-1] = np.moveaxis(iA, 2 - e, 0)[0]
            keep = np.ones((nz, ny, nx))
            for d in (u, w):  # the later axis's faces win on common edges
                k = np.moveaxis(keep, 2 - d, 0)
                k[0], k[-1] = float(not pec(lo[d])), float(not pec(hi[d]))
            tl = tL[c].copy()
            if c in edits:
                tl[-1] = L[c][0]
            self.a.append(t(self.dt * iA * im))
            self.b.append(t(itA * keep))  # without 1/eps
            self.L.append(t(full(L[c], c) * keep))
            self.tL.append(t(full(tl, c)))
        self.bie = [b * self.ie for b in self.b]
        z = lambda: torch.zeros(self.N, dtype=torch.float64, device=self.dev)
        self.E, self.H, self.J = ([z() for _ in range(3)] for _ in range(3))

    def ghosts(self):
        """Before the first step: the last layer of every axis loses its
        tangential H and normal E."""
        nx, ny, nz = self.n
        for a in range(3):
            for c in range(3):
                F = (self.E if c == a else self.H)[c].view(nz, ny, nx)
                F.select(2 - a, self.n[a] - 1).zero_()

    def step(self):
        sh = (1, self.sy, self.sz)
        E, H = self.E, self.H
        e = [E[c] * self.L[c] for c in range(3)]
        for c in range(3):  # H_c -= a_c (d_u e_w - d_w e_u)
            u, w = (c + 1) % 3, (c + 2) % 3
            t = e[u] - e[w]
            t[:-sh[w]] -= e[u][sh[w]:]
            t[:-sh[u]] += e[w][sh[u]:]
            H[c].addcmul_(self.a[c], t, value=-1.0)
        h = [H[c] * self.tL[c] for c in range(3)]
        for c in range(3):
            u, w = (c + 1) % 3, (c + 2) % 3
            t = h[w] - h[u]
            t[sh[w]:] += h[u][:-sh[w]]
            t[sh[u]:] -= h[w][:-sh[u]]
            t *= self.bie[c]
            if self.cond or c == 2:
                t.addcmul_(self.ie, self.J[c], value=-1.0)
            E[c].add_(t, alpha=self.dt)
            if self.cond:
                torch.mul(self.sg, E[c], out=self.J[c])

    def grad_steps(self, beam, line, caps, ie, sg):
        """The same run with 1/eps and sigma per cell as tensors of a gradient."""
        sh = (1, self.sy, self.sz)
        zero = lambda s: torch.zeros(s, dtype=torch.float64, device=self.dev)
        fwd = lambda v, s: torch.cat([v[s:], zero(s)])
        bwd = lambda v, s: torch.cat([zero(s), v[:-s]])
        E, H, out, dtie = list(self.E), list(self.H), [], self.dt * ie
        J = [torch.zeros_like(E[0]) for _ in range(3)]
        take = lambda: torch.stack([E[2][i] for i in caps])
        for n in range(beam.shape[0]):
            out.append(take())
            J[2] = J[2].index_put((line,), beam[n])
            e = [E[c] * self.L[c] for c in range(3)]
            Hn = []
            for c in range(3):
                u, w = (c + 1) % 3, (c + 2) % 3
                Hn.append(H[c] - self.a[c] * (e[u] - fwd(e[u], sh[w]) - e[w] + fwd(e[w], sh[u])))
            H = Hn
            h = [H[c] * self.tL[c] for c in range(3)]
            En = []
            for c in range(3):
                u, w = (c + 1) % 3, (c + 2) % 3
                cu = bwd(h[u], sh[w]) - h[u] - bwd(h[w], sh[u]) + h[w]
                En.append(E[c] + dtie * (self.b[c] * cu - J[c]))
            E = En
            J = [sg * v for v in E]
        return torch.stack(out, dim=1)  # [line][step][z]

    def beam(self, p, steps, ti=None):
        """(flat indices of the beam line, current of every step)."""
        ix, iy = np.abs(self.x - p["xs"]).argmin(), np.abs(self.y - p["ys"]).argmin()
        ti = _ti(p) if ti is None else ti
        n = torch.arange(steps, device=self.dev, dtype=torch.float64)[:, None]
        s = torch.as_tensor(self.z, device=self.dev)[None, :] - C * (n * self.dt)
        s0 = self.z.min() - C * ti
        amp = p["q"] * C / self.dx[ix] / self.dy[iy] / math.sqrt(2 * math.pi * p["sigmaz"] ** 2)
        return self._line(ix, iy), amp * torch.exp(-((s - s0) ** 2) / (2 * p["sigmaz"] ** 2))

    def _line(self, ix, iy):
        return ix + self.sy * iy + self.sz * torch.arange(self.n[2], device=self.dev)

    def window(self, p, plane):
        ix, iy = np.abs(self.x - p["xt"]).argmin(), np.abs(self.y - p["yt"]).argmin()
        if plane == "longitudinal":
            return ix, iy, [self._line(ix, iy)]
        return ix, iy, [self._line(ix + i, iy + j) for i in (-1, 0, 1) for j in (-1, 0, 1)]

    def wake(self, p, wl, plane, freqs=()):
        steps = _steps_of_wl(p, wl)
        line, cur = self.beam(p, steps)
        ix, iy, lines = self.window(p, plane)
        idx = torch.stack(lines)
        cap = torch.zeros((len(lines), steps, self.n[2]), dtype=torch.float64, device=self.dev)
        acc = [torch.zeros((len(freqs), self.N), dtype=torch.complex128, device=self.dev)
               for _ in range(3)] if freqs else None
        for n in range(steps):
            cap[:, n] = self.E[2][idx]
            self.J[2][line] = cur[n]
            self.step()
            for i, f in enumerate(freqs):
                ph = complex(np.exp(-2j * np.pi * f * n * self.dt))
                for c in range(3):
                    acc[c][i] += self.E[c] * ph
        out = _wake_results(self, p, wl, plane, cap, ix, iy)
        nx, ny, nz = self.n
        if freqs:
            for c, k in enumerate(("Ex", "Ey", "Ez")):
                out[k] = acc[c].view(len(freqs), nz, ny, nx).permute(0, 3, 2, 1)
        return out


def _wake_axes(sim, p, wl, steps):
    """Time and s axes of a run (their spacing has the field dtype's dt)."""
    dt = np.dtype(p["dtype"]).type(sim.dt)
    t = np.arange(0, steps * dt, dt)
    dts = t[2] - t[1]
    return t, dts, np.arange(-_ti(p) * C, wl, dts * C)


def _line_integrals(sim, p, cap, t, dts, s):
    """WP of every captured line [line][s]: each line's integral is added to
    the line before it, then divided by the charge."""
    zf, k0 = sim.z, p["skip"]
    z, nt = zf[k0:len(zf) - k0], min(len(t), cap.shape[1])
    ncols = nt if len(cap) == 1 else len(t)
    tt = lambda v: torch.as_tensor(np.asarray(v, dtype=np.float64), device=sim.dev)
    ts = (tt(z)[None, :] + tt(s)[:, None]) / C
    ts = ts - float(zf.min() / C)
    ts = ts - float(t[0])
    ts = ts + _ti(p)
    it = torch.trunc(ts / float(dts)).to(torch.int64)
    col = torch.where(it < 0, it + ncols, it)
    ok = (it < nt) & (col >= 0) & (col < nt)
    k = torch.arange(k0, k0 + len(z), device=sim.dev)[None, :]
    dz = tt(sim.dz[:len(z)])[None, :]
    out, run = [], torch.zeros(len(s), dtype=torch.float64, device=sim.dev)
    for line in cap:
        g = torch.where(ok, line[col.clamp(0, nt - 1), k], torch.zeros_like(ts)) * dz
        run = (run + g.sum(1)) / (p["q"] * 1e12)
        out.append(run)
    return torch.stack(out)


def _dft(sim, sig, s, fmax, samples=1001):
    ds = np.mean(s[1:] - s[:-1])
    N = int((C / ds) // fmax * samples)
    f = np.fft.fftfreq(N, ds / C)
    keep = np.logical_and(f >= 0, f < fmax)
    return f[keep], ds, np.fft.fft(sig, n=N)[keep]


def _wake_results(sim, p, wl, plane, cap, ix, iy):
    t, dts, s = _wake_axes(sim, p, wl, cap.shape[1])
    W = _line_integrals(sim, p, cap, t, dts, s).cpu().numpy()
    WP = W[len(W) // 2]
    lam = np.exp(-(s ** 2) / (2 * p["sigmaz"] ** 2)) / (p["sigmaz"] * np.sqrt(2 * np.pi))
    fmax = C / (3.0 * p["sigmaz"])
    f, ds, lf = _dft(sim, lam * C, s, fmax)
    out = dict(s=s, WP=WP, f=f, Z=-_dft(sim, WP * 1e12, s, fmax)[2] / lf,
               loss=float(-math.fsum(WP * lam) * (s[2] - s[1])))
    if plane == "both":
        xf, yf = sim.x[ix - 1:ix + 2], sim.y[iy - 1:iy + 2]
        d = s[2] - s[1]
        I = np.concatenate([np.zeros((9, 1)), np.cumsum(W, axis=1)[:, :-1]], axis=1) * d
        WPx = -(I[7] - I[1]) / (xf[2] - xf[0])
        WPy = -(I[5] - I[3]) / (yf[2] - yf[0])
        out.update(WP_3d=W.reshape(3, 3, -1), WPx=WPx, WPy=WPy,
                   Zx=1j * _dft(sim, WPx * 1e12, s, fmax)[2] / lf,
                   Zy=1j * _dft(sim, WPy * 1e12, s, fmax)[2] / lf)
    return out


def _exact_adjoint(case, seed):
    p = _adjoint_structure(case, seed)
    sim = _Sim(p)
    wl = case["wl"]
    steps = _steps_of_wl(p, wl)
    er, sg = (torch.tensor(v, device=sim.dev, requires_grad=True)
              for v in _block_values(case, seed))
    reg = _block_region(case)
    nx, ny, nz = sim.n
    blk = (slice(*reg[2]), slice(*reg[1]), slice(*reg[0]))
    ie, sf = sim.ie.view(nz, ny, nx).clone(), sim.sg.view(nz, ny, nx).clone()
    ie[blk] = (1 / (er * EPS0)).permute(2, 1, 0)
    sf[blk] = sg.permute(2, 1, 0)
    line, cur = sim.beam(p, steps)
    _, _, caps = sim.window(p, "both")
    cap = sim.grad_steps(cur, line, caps, ie.reshape(-1), sf.reshape(-1))
    t, dts, s = _wake_axes(sim, p, wl, steps)
    WP = _line_integrals(sim, p, cap, t, dts, s)[4]
    lam = torch.as_tensor(np.exp(-(s ** 2) / (2 * p["sigmaz"] ** 2))
                          / (p["sigmaz"] * np.sqrt(2 * np.pi)), device=sim.dev)
    ds = np.mean(s[1:] - s[:-1])
    fmax = C / (3.0 * p["sigmaz"])
    N = int((C / ds) // fmax * 1001)
    f = np.fft.fftfreq(N, ds / C)
    band = torch.as_tensor(np.nonzero((f >= 0) & (f < min(fmax, 3e9)))[0], device=sim.dev)
    Z = -torch.fft.fft(WP * 1e12, n=N)[band] / torch.fft.fft(lam * C, n=N)[band]
    L = -(WP * lam).sum() * (s[2] - s[1]) + 1e-13 * (Z.abs() ** 2).sum() * (f[1] - f[0])
    L.backward()
    return dict(L=float(L.detach()), g_eps=er.grad, g_sigma=sg.grad)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        ps = _batch_structures(case, seed)
        if sum(_steps_of_wl(p, w) for p, w in ps) > 25000:
            return None
        outs, E, H = [], [], []
        for p, w in ps:
            sim = _Sim(p)
            outs.append(sim.wake(p, w, "both"))
            E.append(torch.cat(sim.E))
            H.append(torch.cat(sim.H))
        return dict(_join(outs), E=E, H=H)
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "adjoint":  # every step's states are kept for the gradient
        steps = _steps_of_wl(_structure_axes(case), case["wl"])
        return None if n * steps * 80 > 1.0e11 else _exact_adjoint(case, seed)
    if kind == "emsolve":
        return _exact_emsolve(case, seed)
    p = _structure(case, seed)
    sim = None
    if kind == "loop":
        sim = _Sim(p)
        line, cur = sim.beam(p, case["steps"], ti=2.0 * p["sigmaz"] / C)
        for i in range(case["steps"]):
            sim.J[2][line] = cur[i]
            sim.step()
        return dict(E=torch.cat(sim.E), H=torch.cat(sim.H))
    if kind == "post":
        return _Sim(p).wake(p, _wl_for_steps(p, case["steps"]), "both")
    if n * _steps_of_wl(p, case["wl"]) > EXACT_MAX_CELL_STEPS:
        return None
    sim = _Sim(p)
    out = sim.wake(p, case["wl"], case["plane"], [1.1e9 + 0.9e9 * i for i in range(case["nfreq"])])
    out.update(E=torch.cat(sim.E), H=torch.cat(sim.H))
    return out


def _exact_emsolve(case, seed):
    sim = _Sim(_em_structure(case))
    w = _plane_wave(case, seed)
    nx, ny, nz = sim.n
    plane = slice(w["zs"] * sim.sz, (w["zs"] + 1) * sim.sz)
    om = 2 * np.pi * w["f"]
    for n in range(case["steps"]):
        t = n * sim.dt
        on = 1.0 if t <= w["nodes"] / w["f"] else 0.0
        cw = on * w["amplitude"] * math.cos(om * t + w["phase"])
        sim.H[1][plane] = -cw
        sim.E[0][plane] = cw / ((om / C) / (MU0 * C))
        if n == 0:
            sim.ghosts()
        sim.step()
        if case["top"] == "abc":
            for F in sim.E + sim.H:
                F[:sim.sz] = F[sim.sz:2 * sim.sz]
    return dict(E=torch.cat(sim.E), H=torch.cat(sim.H), J=torch.cat(sim.J))
