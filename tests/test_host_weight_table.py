"""CPU: when the weight table of the two-step kernel is made, and what a failure
while it is made leaves behind (SolverFIT3D._weight_table, _prepare_fused).

The solver is built on CPU tensors; the library's two table kernels are replaced
by a stand-in that marks every class of every material as used.
"""

import ctypes

import numpy as np
import pytest
import torch

import wakis_amd as wa
import wakis_amd.field as wf
from wakis_amd import _lib


class _Kernels:
    """wf_weight_rows and wf_weight_codes on host memory."""

    def __init__(self):
        self.calls, self.fail = [], None

    def wf_weight_rows(self, h, code, mat, nmat, metric, dt, rows, used, st):
        self.calls.append("rows")
        nk = 27 * nmat
        r = np.ctypeslib.as_array(ctypes.cast(rows, ctypes.POINTER(ctypes.c_int32)),
                                  (nk * _lib.WF_WEIGHT_ROW,))
        r[:] = np.arange(nk * _lib.WF_WEIGHT_ROW)
        u = np.ctypeslib.as_array(ctypes.cast(used, ctypes.POINTER(ctypes.c_int32)), (nk + 1,))
        u[:] = 1
        u[nk] = 0
        return 0

    def wf_weight_codes(self, h, code, nmat, row_of, wcode, st):
        self.calls.append("codes")
        if self.fail is not None:
            raise self.fail
        return 0


@pytest.fixture
def kernels(monkeypatch):
    k = _Kernels()
    monkeypatch.setattr(wf, "default_device", lambda: torch.device("cpu"))
    monkeypatch.setattr(wa.SolverFIT3D, "_create_handle", lambda self, lib: None)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a, **kw: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(_lib, "lib", lambda: k)
    monkeypatch.setattr(_lib, "stream_ptr", lambda *a: None)
    return k


def _solver(dtype=np.float32):
    x = np.linspace(-4e-3, 4e-3, 9)
    blk = np.zeros((8, 8, 8), dtype=bool)
    blk[2:5, 2:5, 2:5] = True
    grid = wa.GridFIT3D(x=x, y=x, z=x, stl_solids={"b": blk}, stl_materials={"b": [3.0, 1.0]},
                        verbose=0)
    s = wa.SolverFIT3D(grid, bc_low=["pec"] * 3, bc_high=["pec"] * 3, use_stl=True, bg=[1.0, 1.0],
                       dtype=dtype, verbose=0)
    s._handle = None
    s._beam_line = (4, 4)
    return s


def _args(s, nsteps=100):
    a = s._step_args(nsteps)
    a.jmode, a.beam_table = _lib.WF_J_LINE, 8
    return a


@pytest.mark.parametrize("where", ["codes", "as_tensor"])
def test_no_half_made_table_after_an_exception(kernels, monkeypatch, where):
    s = _solver()
    assert s._material_table()
    if where == "codes":
        kernels.fail = KeyboardInterrupt()
    else:
        def interrupted(*a, **kw):
            raise KeyboardInterrupt
        monkeypatch.setattr(torch, "as_tensor", interrupted)
    with pytest.raises(KeyboardInterrupt):
        s._weight_table()
    assert s._wcode is None and s._wtab is None and s._wkey is None


def test_table_made_after_an_interrupted_attempt(kernels):
    s = _solver()
    assert s._material_table()
    kernels.fail = KeyboardInterrupt()
    with pytest.raises(KeyboardInterrupt):
        s._weight_table()
    kernels.fail = None
    assert s._weight_table()
    assert s._wcode.shape == (s.N,) and s._wtab.shape == (1 + 27 * s._nmat, _lib.WF_WEIGHT_ROW)


def test_run_goes_on_without_memory_for_the_table(kernels, monkeypatch):
    s = _solver()
    empty = torch.empty

    def full(*a, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("out of memory")
        return empty(*a, **kw)
    monkeypatch.setattr(torch, "empty", full)
    a = _args(s)
    assert s._prepare_fused(a)
    assert a.code and not a.wcode and a.nw == 0
    n = len(kernels.calls)
    assert s._prepare_fused(_args(s)) and len(kernels.calls) == n  # not tried again


def _no_pairs():
    """Calls that run one step per launch."""
    yield "trajectory", dict(traj_E=8)
    yield "box", dict(box_hi=(3, 3, 3))
    yield "monitor without scratch", dict(mon_acc=8)
    yield "no beam table", dict(beam_table=None)
    for name, v in (("fused_variant", 1), ("fused_full_rows", 2), ("fused_cells_per_lane", 1),
                    ("fused_two_step", 0), ("skip_masks", False)):
        yield name, {name: v}


def test_no_table_for_calls_of_single_steps(kernels):
    s = _solver()
    for name, kw in _no_pairs():
        a, held = _args(s), {}
        for k, v in kw.items():
            if hasattr(s, k):
                held[k] = getattr(s, k)
                setattr(s, k, v)
            elif isinstance(v, tuple):
                getattr(a, k)[:] = v
            else:
                setattr(a, k, v)
        assert s._prepare_fused(a) and a.code and not a.wcode, name
        for k, v in held.items():
            setattr(s, k, v)
    assert kernels.calls == []
    short = _args(s, 40)
    assert s._prepare_fused(short) and not short.wcode and kernels.calls == []
    a = _args(s)
    assert s._prepare_fused(a) and a.wcode and kernels.calls == ["rows", "codes"]
    short = _args(s, 40)  # made already
    assert s._prepare_fused(short) and short.wcode and kernels.calls == ["rows", "codes"]
    s.ieps[2:5, 2:5, 2:5, "x"] = 1e10  # new materials: again by the first longer call
    s.update_tensors()
    short = _args(s, 40)
    assert s._prepare_fused(short) and not short.wcode and kernels.calls == ["rows", "codes"]
    a = _args(s)
    assert s._prepare_fused(a) and a.wcode and len(kernels.calls) == 4
