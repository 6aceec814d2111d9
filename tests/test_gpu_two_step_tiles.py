"""GPU: tiles of the two-step kernel (k_fused4_t2) on rows of any length.

Calls of several steps on grids whose rows are no whole number of lanes, longer
than 256 cells (several tiles along x), shorter than a lane or exactly whole
waves, with and without conduction, FP32 and FP64: E, H, J and the captured Ez
window bitwise those of one step per launch, whose results other tests tie to
the oracle. The spare buffers hold the fields one step back afterwards, so
energy() works as after single steps.
"""

import numpy as np
import pytest
import torch

from tests.test_gpu_two_step import _beam_setup, _cavity_solver, _pillbox_solver

pytestmark = pytest.mark.gpu


def _run(make, dims, dtype, two_step, chunks, kz):
    s = make(dims, two_step, kz, dtype)
    args, cap = _beam_setup(s, sum(chunks))
    n0, pairs = 0, []
    for k in chunks:
        s._run(args(n0, k))
        assert s.last_path == "fused"
        pairs.append(s.last_pairs)
        n0 += k
    torch.cuda.synchronize()
    return ([s.E.to_numpy(), s.H.to_numpy(), s.J.to_numpy(), cap.cpu().numpy()], pairs, s)


@pytest.mark.parametrize("make", [_cavity_solver, _pillbox_solver])
@pytest.mark.parametrize("dims,chunks,kz", [
    ((41, 13, 40), (9, 4), 0),     # one cell in the last lane
    ((43, 40, 33), (3, 6), 1),     # one plane per chunk
    ((128, 17, 40), (7,), 0),      # whole rows of lanes, not of waves
    ((255, 9, 30), (8,), 0),       # FP32: a cut lane in a whole wave's row
    ((252, 12, 30), (5,), 7),
    ((257, 12, 30), (5,), 0),      # one cell past 256
    ((300, 40, 30), (5, 4), 0),    # tiles along x
    ((517, 7, 29), (6,), 4),
    ((36, 300, 28), (4,), 0),      # many short rows
])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_pairs_equal_single_steps(make, dims, chunks, kz, dtype):
    print("pairs", make.__name__, dims, chunks, kz, np.dtype(dtype).name, flush=True)
    ref, _, s1 = _run(make, dims, dtype, 0, chunks, kz)
    got, pairs, s2 = _run(make, dims, dtype, 1, chunks, kz)
    assert all(pairs) and not s2.last_two_step
    assert np.any(ref[0] != 0) and np.any(ref[3] != 0)
    for name, r, g in zip(("E", "H", "J", "capture"), ref, got):
        assert np.array_equal(g, r), f"{name} differs ({np.count_nonzero(g != r)} values)"
    assert s1.energy() == s2.energy()


def test_two_steps_are_not_paired():
    """A call of one or two steps has no pair before its single last steps."""
    for k in (1, 2):
        _, pairs, _ = _run(_cavity_solver, (41, 13, 40), np.float32, 1, (k,), 0)
        assert pairs == [False]
