"""Flux reductions and the band increment at the edges of their loops: column-layer counts that are and are
not whole 16-byte vectors, bands of 1 to 33 g-points (the reduction loads 8 at a time), one direct flux more
or less, and bands that do not follow each other.

Sums are compared bit for bit with sums in g-point order in the same type.  Each increment output is a sum
of two products over a sum, a few roundings each, of positive terms: 8 eps.
"""
import copy
import ctypes as C

import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_adjoint import G, _host                           # noqa: F401  (G is a fixture)
from test_gpu_gas_optics_adjoint import ragged

pytestmark = pytest.mark.gpu


def _kdist(syn, precision, order=None):
    from rrtmgp_amd import api
    k = ragged(syn.make_kdist(False, 12))
    if order is not None:
        k = copy.deepcopy(k)
        k.band2gpt = np.asfortranarray(k.band2gpt[:, order])
    return api.KDist(k, AVAILABLE, precision)


def _in_order(f):
    s = f[..., 0].copy()
    for g in range(1, f.shape[-1]):
        s += f[..., g]
    return s


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("ncol,nlev,order", [(1, 1, None), (3, 5, None), (64, 4, None), (257, 3, None),
                                             (5, 3, [1, 0, 2, 3, 5, 4])])
def test_reduce(G, syn, precision, ncol, nlev, order):
    dt = G.real_dtype(precision)
    kd = _kdist(syn, precision, order)
    lims = kd.band_lims.T
    rng = np.random.default_rng(ncol)
    up, dn, dr = (rng.uniform(0, 10, (ncol, nlev, kd.ngpt)).astype(dt) for _ in range(3))
    dev = G.DeviceArray.from_host
    for direct in (False, True):
        for byband in (False, True):
            o = {k: _host(v) for k, v in G.fluxes_reduce(kd, dev(up), dev(dn), dev(dr) if direct else None,
                                                         byband=byband).items()}
            want = {"flux_up": _in_order(up), "flux_dn": _in_order(dn)}
            want["flux_net"] = want["flux_dn"] - want["flux_up"]
            if direct:
                want["flux_dn_dir"] = _in_order(dr)
            if byband:
                bands = lambda f: np.stack([_in_order(f[:, :, a - 1:b]) for a, b in lims], 2)   # noqa: E731
                want.update({"bnd_flux_up": bands(up), "bnd_flux_dn": bands(dn)})
                want["bnd_flux_net"] = want["bnd_flux_dn"] - want["bnd_flux_up"]
                if direct:
                    want["bnd_flux_dn_dir"] = bands(dr)
            assert o.keys() == want.keys()
            for k in want:
                assert np.array_equal(o[k], want[k]), (k, direct, byband)


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("ncol,nlay", [(1, 1), (3, 5), (64, 4), (257, 3), (130, 9)])
def test_increment_by_band(G, syn, precision, ncol, nlay):
    dt = G.real_dtype(precision)
    kd = _kdist(syn, precision)
    lims = kd.band_lims.T
    band = np.concatenate([np.full(b - a + 1, i) for i, (a, b) in enumerate(lims)])
    rng = np.random.default_rng(ncol)
    t1, s1, g1 = (rng.uniform(0, 1, (ncol, nlay, kd.ngpt)).astype(dt) for _ in range(3))
    t2, s2, g2 = (rng.uniform(0, 1, (ncol, nlay, kd.nbnd)).astype(dt) for _ in range(3))
    t2[rng.random(t2.shape) < 0.5] = 0
    dev = G.DeviceArray.from_host
    a, b, c, x, y, z = (v.astype(np.float64) for v in (t1, s1, g1, t2[:, :, band], s2[:, :, band], g2[:, :, band]))
    tol = 8 * np.finfo(dt).eps
    d = dev(t1)
    G.add_to(kd, d, dev(t2))
    np.testing.assert_allclose(_host(d), a + x, rtol=tol)
    d, ds, dg = dev(t1), dev(s1), dev(g1)
    G.add_to(kd, d, dev(t2), ds, dg, dev(s2), dev(g2))
    np.testing.assert_allclose(_host(d), a + x, rtol=tol)
    np.testing.assert_allclose(_host(ds), (a * b + x * y) / (a + x), rtol=tol)
    np.testing.assert_allclose(_host(dg), (a * b * c + x * y * z) / (a * b + x * y), rtol=tol)


@pytest.mark.parametrize("ncol,nlay", [(1639, 31), (1, 49151), (49153, 1)])
def test_increment_of_large_odd_slices(G, syn, ncol, nlay):
    """FP64 two-stream increments beyond the size from which a thread takes an element of the whole array, with
    bands that leave g-points out and overlap; bit for bit what a slice of fewer elements gives."""
    from rrtmgp_amd import _lib
    dt, ng = np.float64, 9
    lims = np.array([[1, 3], [3, 4], [6, 9]], dtype=np.int32)
    rng = np.random.default_rng(ncol)
    n = ncol * nlay
    a = [rng.uniform(0, 1, (n, ng)) for _ in range(3)]
    b = [rng.uniform(0, 1, (n, len(lims))) for _ in range(3)]
    dev = lambda x, t=dt: G.DeviceArray.from_host(np.asfortranarray(x), t)               # noqa: E731
    for name in ("inc_bybnd", "inc_bybnd_coalbedo"):
        def run(part):
            x, y = [dev(v[part]) for v in a], [dev(v[part]) for v in b]
            m, lim = len(a[0][part]), dev(lims.ravel(), np.int32)
            _lib.check_hip(getattr(_lib.hip(), f"rrtmgp_hip_{name}_f64")(
                C.c_int64(m), C.c_int64(1), C.c_int64(ng), *[v.ptr for v in x + y], C.c_int64(len(lims)), lim.ptr, None))
            return [_host(v) for v in x]

        whole = run(slice(None))
        for s in (slice(0, 999), slice(n - 999, n)):
            for w, p in zip(whole, run(s)):
                assert np.array_equal(w[s], p), name
        assert np.array_equal(whole[0][:, 4], a[0][:, 4])                # of no band
