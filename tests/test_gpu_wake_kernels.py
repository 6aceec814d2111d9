"""GPU: the wake kernels at the edges of their tiles.

* ``wf_wake_wp`` (16 samples of s per workgroup, 128 rows per chunk, the columns
  kept in LDS up to 1,800 rows): bitwise the reference's loop (wakeSolver.py:
  485-537) written out in numpy, one multiplication and addition per row in
  order, the running value carried from line to line.
* ``wf_wake_trans`` (one wave per prefix sum): bitwise numpy's own sums of
  WP[:n] (wakeSolver.py:583-612), across the tree's leaves and its 8,192-value
  blocks.
* ``wf_dft`` (up to four signals per launch): against the direct sum in numpy's
  long double. A bin's error is bounded by the rounding of the phase, the
  sine and cosine (2 ulp each) and the product: 4 eps sum |x| is twice that.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _ref_wp(cap, z, dz, s, v, zref_v, t0, ti, dt, nt, ncols, qe12, cm, k0):
    """[line][s], the reference's loop."""
    nz = len(z)
    out = np.zeros((cap.shape[0], len(s)))
    acc = np.zeros(len(s))
    for l in range(cap.shape[0]):
        for k in range(nz):
            kr = nz - 1 - k if cm else k
            ts = (z[kr] - s) / (-v) if cm else (z[kr] + s) / v
            ts = ts - zref_v - t0 + ti
            it = (ts / dt).astype(np.int64)
            col = np.where(it < 0, it + ncols, it)
            ok = (it < nt) & (col >= 0) & (col < nt)
            e = np.where(ok, cap[l, np.clip(col, 0, nt - 1), k0 + kr].astype(np.float64), 0.0)
            acc = acc + np.where(ok, e * (-dz[k] if cm else dz[k]), 0.0)
        acc = acc / qe12
        out[l] = acc
    return out


@pytest.mark.parametrize("nz,ns,nlines", [(1, 1, 1), (2, 15, 9), (127, 16, 9), (128, 17, 1),
                                          (129, 40, 9), (300, 33, 9), (1800, 20, 1),
                                          (1801, 20, 2)])
@pytest.mark.parametrize("cm", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_line_integrals_match_the_loop(nz, ns, nlines, cm, dtype):
    from wakis_amd import _lib
    print("wake wp", nz, ns, nlines, cm, np.dtype(dtype).name, flush=True)
    rng = np.random.default_rng(nz + ns)
    k0, Nz, nt, ncols = 2, nz + 5, 57, 59
    cap = rng.standard_normal((nlines, nt + 3, Nz)).astype(dtype)
    z = np.cumsum(rng.uniform(0.5, 1.5, nz))
    dz = rng.uniform(0.5, 1.5, nz)
    v, dt, t0, ti, qe12 = 2.0, max(nz, 8) / 60.0, 0.1, 0.3, 3.7
    s = np.linspace(-3.0, 0.6 * nz + 2, ns)
    zref_v = z.max() / (-v) if cm else z.min() / v
    ref = _ref_wp(cap, z, dz, s, v, zref_v, t0, ti, dt, nt, ncols, qe12, cm, k0)
    d = [_dev(a) for a in (cap, z, dz, s)]
    out = torch.full((nlines, ns), np.nan, dtype=torch.float64, device="cuda")
    _lib.check(_lib.lib().wf_wake_wp(
        _lib.ptr(d[0]), _lib.WF_F64 if dtype == np.float64 else _lib.WF_F32, nlines, nt + 3, Nz,
        k0, nz, _lib.ptr(d[1]), _lib.ptr(d[2]), _lib.ptr(d[3]), ns, v, zref_v, t0, ti, dt, nt,
        ncols, int(cm), qe12, _lib.ptr(out), _lib.stream_ptr()), "wf_wake_wp")
    assert np.any(ref != 0)
    assert np.array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize("ns", [1, 2, 7, 9, 129, 137, 300, 1100, 8300, 16500])
def test_prefix_sums_are_numpys(ns):
    from wakis_amd import _lib
    print("wake trans", ns, flush=True)
    rng = np.random.default_rng(ns)
    W = rng.standard_normal((9, ns)) * 10.0 ** rng.uniform(-6, 6, (9, ns))
    ds, dx, dy = 0.3, 1.7, 0.9
    d = _dev(W)
    px, py = (torch.full((ns,), np.nan, dtype=torch.float64, device="cuda") for _ in range(2))
    _lib.check(_lib.lib().wf_wake_trans(_lib.ptr(d), ns, ds, dx, dy, _lib.ptr(px), _lib.ptr(py),
                                        _lib.stream_ptr()), "wf_wake_trans")
    I = lambda l, n: np.sum(W[l, :n]) * ds
    pick = range(ns) if ns < 2000 else list(range(0, 300)) + list(range(ns - 400, ns)) + [8191, 8192]
    gx, gy = px.cpu().numpy(), py.cpu().numpy()
    for n in pick:
        assert gx[n] == -(I(7, n) - I(1, n)) / dx, n
        assert gy[n] == -(I(5, n) - I(3, n)) / dy, n


@pytest.mark.parametrize("nsig", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("length,N,nbins", [(1, 7, 3), (255, 1001, 40), (257, 257, 257),
                                            (3000, 4097, 65)])
def test_dft_bins(nsig, length, N, nbins):
    from wakis_amd import _lib
    print("dft", nsig, length, N, nbins, flush=True)
    rng = np.random.default_rng(length)
    x = rng.standard_normal((nsig, length))
    d = _dev(x)
    out = torch.full((nsig, nbins, 2), np.nan, dtype=torch.float64, device="cuda")
    _lib.check(_lib.lib().wf_dft(_lib.ptr(d), nsig, length, N, nbins, _lib.ptr(out),
                                 _lib.stream_ptr()), "wf_dft")
    ph = (np.arange(nbins)[:, None] * np.arange(length)[None, :] % N).astype(np.longdouble)
    ang = -2 * np.longdouble("3.14159265358979323846264338327950288") * ph / N
    ref = np.stack([x.astype(np.longdouble) @ np.cos(ang).T,
                    x.astype(np.longdouble) @ np.sin(ang).T], axis=2)
    err = np.abs(out.cpu().numpy() - ref)
    bound = 4 * np.finfo(np.float64).eps * np.abs(x).sum(axis=1)[:, None, None]
    assert np.all(err <= bound), float((err / bound).max())
