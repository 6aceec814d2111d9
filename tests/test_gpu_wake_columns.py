"""GPU: line integrals on both sides of the rule that keeps the columns of a line in
LDS (wp_keep_columns): several lines, and at most one workgroup of 16 samples per CU
where more than 768 rows hold a CU to one. Bitwise the loop written out in numpy, at
about 300 samples spread over the launch."""

import numpy as np
import pytest
import torch

from tests.test_gpu_wake_kernels import _dev, _ref_wp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,ns,nlines", [(768, 16 * 300, 2), (769, 16 * 300, 2), (769, 16 * 256, 2),
                                          (769, 16 * 256 + 1, 2), (1800, 20, 3), (1801, 20, 3),
                                          (300, 16 * 300, 1)])
@pytest.mark.parametrize("cm", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_line_integrals_on_both_sides_of_the_rule(nz, ns, nlines, cm, dtype):
    from wakis_amd import _lib
    print("wake columns", nz, ns, nlines, cm, np.dtype(dtype).name, flush=True)
    rng = np.random.default_rng(nz + ns)
    k0, Nz, nt = 1, nz + 2, 61
    cap = rng.standard_normal((nlines, nt, Nz)).astype(dtype)
    z = np.cumsum(rng.uniform(0.5, 1.5, nz))
    dz = rng.uniform(0.5, 1.5, nz)
    v, dt, t0, ti, qe12 = 2.0, nz / 60.0, 0.1, 0.3, 3.7
    s = np.linspace(-3.0, 0.6 * nz, ns)
    zref_v = z.max() / (-v) if cm else z.min() / v
    pick = np.arange(0, ns, max(1, ns // 300))
    ref = _ref_wp(cap, z, dz, s[pick], v, zref_v, t0, ti, dt, nt, nt, qe12, cm, k0)
    d = [_dev(a) for a in (cap, z, dz, s)]
    out = torch.full((nlines, ns), np.nan, dtype=torch.float64, device="cuda")
    _lib.check(_lib.lib().wf_wake_wp(
        _lib.ptr(d[0]), _lib.WF_F64 if dtype == np.float64 else _lib.WF_F32, nlines, nt, Nz, k0,
        nz, _lib.ptr(d[1]), _lib.ptr(d[2]), _lib.ptr(d[3]), ns, v, zref_v, t0, ti, dt, nt, nt,
        int(cm), qe12, _lib.ptr(out), _lib.stream_ptr()), "wf_wake_wp")
    got = out.cpu().numpy()
    assert np.any(ref != 0) and np.isfinite(got).all()
    assert np.array_equal(got[:, pick], ref)
