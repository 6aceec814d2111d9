"""GPU: weight codes of grids with other boundaries than PEC: the face classes hold
the folded products, and pairs on them leave the fields as single steps do."""

import numpy as np
import pytest
import torch

from tests import test_gpu_weight_codes as wc
from tests.test_gpu_two_step import _beam_setup

pytestmark = pytest.mark.gpu

# (faces, whether pairs apply: the flat-index wrap terms of the others are live)
BCS = [(("pmc", "pmc", "pmc"), True), (("pec", "pmc", "pml"), True), (("pec", "pec", "pml"), True),
       (("pec", "pec", "pmc"), True), (("periodic", "periodic", "periodic"), False),
       (("pmc", "pec", "abc"), False), (("abc", "abc", "abc"), False),
       (("periodic", "pec", "pml"), False)]


@pytest.mark.parametrize("bc,pairs", BCS)
@pytest.mark.parametrize("dims", [(41, 24, 33), (64, 14, 40)])
def test_rows_and_pairs(bc, pairs, dims):
    print("weight codes", bc, dims, flush=True)

    def make(d, two_step):
        return wc._insert_solver(d, two_step, bc=bc)
    wc.test_rows_hold_the_folded_products(make, dims)
    out = []
    for two_step in (0, 8):
        s = make(dims, two_step)
        assert s._material_table() and s._weight_table()
        args, cap = _beam_setup(s, 10)
        a = args(0, 10)
        s._run(a)
        assert s.last_pairs == bool(two_step and pairs)
        assert s.last_path == ("fused" if pairs else "general")
        out.append((s, cap))
    assert bool((out[0][0].E.array != 0).any())
    for name in ("E", "H", "J"):
        assert torch.equal(getattr(out[0][0], name).array, getattr(out[1][0], name).array), name
    assert torch.equal(out[0][1], out[1][1]) and np.isfinite(out[0][1].cpu().numpy()).all()
