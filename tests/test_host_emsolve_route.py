"""CPU: emsolve takes a solver's own one_step (a subclass's, or one set on the
object) at every step instead of the library's loop."""

from types import MethodType

import numpy as np
import pytest
import torch

import wakis_amd as wa
import wakis_amd.field as wf
from wakis_amd import _lib


class Counting(wa.SolverFIT3D):
    steps = 0

    def one_step(self):
        self.steps += 1


@pytest.mark.parametrize("on_object", [True, False])
def test_own_one_step_is_called_at_every_step(monkeypatch, on_object):
    monkeypatch.setattr(wf, "default_device", lambda: torch.device("cpu"))
    monkeypatch.setattr(wa.SolverFIT3D, "_create_handle", lambda self, lib: None)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a, **kw: None)
    x = np.linspace(0, 8e-3, 9)
    s = (wa.SolverFIT3D if on_object else Counting)(
        wa.GridFIT3D(x=x, y=x, z=x, verbose=0), bc_low=["pec"] * 3, bc_high=["pec"] * 3,
        bg=[1.0, 1.0, 0.3], dtype=np.float32, verbose=0)
    s._handle = None
    monkeypatch.setattr(_lib, "lib", lambda: pytest.fail("the library's loop was called"))
    if on_object:
        s.steps = 0
        s.one_step = MethodType(Counting.one_step, s)
    s.emsolve(20, source=wa.PlaneWave(f=1e9, zs=4))
    assert s.steps == 20
