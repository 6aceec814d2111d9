"""GPU: forms of the two-step kernel that only large grids and calls ending in a pair
reach, bitwise against one step per launch.

FP32 stores streamed past the caches (above 4.17 million cells, rows of whole
128-byte lines): on material and weight codes, with and without conduction, and
of the first step's E for a field monitor. J = sigma E stored by the last pair of
a call on weight codes.
"""

import numpy as np
import pytest
import torch

from tests.test_gpu_two_step import _beam_setup, _cavity_solver, _pillbox_solver

pytestmark = pytest.mark.gpu

STREAMED = (256, 128, 136)
assert 48 * np.prod(STREAMED) > 200e6


def _steps(make, dims, two_step, chunks, codes):
    s = make(dims, two_step)
    s.use_weight_codes = codes
    if two_step and codes:
        assert s._material_table() and s._weight_table()
    args, cap = _beam_setup(s, sum(chunks))
    n0 = 0
    for k in chunks:
        a = args(n0, k)
        s._run(a)
        assert bool(a.wcode) == bool(two_step and codes)
        n0 += k
    return s, cap


def _same(s1, cap1, s2, cap2):
    assert bool((s1.E.array != 0).any())
    for name in ("E", "H", "J"):
        assert torch.equal(getattr(s1, name).array, getattr(s2, name).array), name
    assert torch.equal(cap1, cap2) and bool((cap1 != 0).any())


@pytest.mark.parametrize("make", [_cavity_solver, _pillbox_solver])
@pytest.mark.parametrize("codes", [True, False])
@pytest.mark.parametrize("dims,two_step,chunks", [
    (STREAMED, 1, (6, 4)), (STREAMED, 8, (5, 2)),
    ((40, 13, 40), 8, (8, 6)), ((64, 64, 24), 8, (2, 4)), ((256, 9, 30), 4, (10,))])
def test_calls_that_end_with_a_pair(make, codes, dims, two_step, chunks):
    print("pair at the end", make.__name__, codes, dims, two_step, chunks, flush=True)
    s1, c1 = _steps(make, dims, 0, chunks, codes)
    s2, c2 = _steps(make, dims, two_step, chunks, codes)
    assert s2.last_two_step and chunks[-1] % 2 == 0
    _same(s1, c1, s2, c2)
    if make is _pillbox_solver:
        assert torch.equal(s2.J.array[:2 * s2.N], (s2.sigma.array * s2.E.array)[:2 * s2.N])


@pytest.mark.parametrize("make", [_cavity_solver, _pillbox_solver])
@pytest.mark.parametrize("codes", [True, False])
def test_monitor_with_streamed_stores(make, codes):
    from wakis_amd import FieldMonitor, _lib
    print("monitor, streamed", make.__name__, codes, flush=True)
    out = []
    for two_step in (0, 1):
        s = make(STREAMED, two_step)
        s.use_weight_codes = codes
        if two_step and codes:
            assert s._material_table() and s._weight_table()
        args, cap = _beam_setup(s, 12)
        m = FieldMonitor([1e9, 3e9])
        work = s._monitor_work()
        for n0, k in ((0, 9), (9, 3)):
            a = args(n0, k)
            keep = m._step_args(a, s.E, s.dt, k)
            if two_step:
                a.mon_work, a.mon_slots = _lib.ptr(work), work.shape[0]
            s._run(a)
            assert s.last_pairs == bool(two_step)
            m.time_index += k
            del keep
        out.append((s, cap, m.get_components()))
    _same(out[0][0], out[0][1], out[1][0], out[1][1])
    for c in ("Ex", "Ey", "Ez"):
        a, b = out[0][2][c], out[1][2][c]
        assert torch.equal(a, b) and bool((b != 0).any()), c
