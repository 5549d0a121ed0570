"""Scratch of the adjoint drivers, and the solver adjoints that write cotangents over their inputs."""
import ctypes as C

import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_adjoint import G, _host                           # noqa: F401  (G is a fixture)

pytestmark = pytest.mark.gpu


def test_peak_scratch(G, syn, kd_lw, kd_sw, lut_lw, lut_sw):
    """Both drivers at 16384 x 128 in FP32, all-sky, leave at most 3.1 GB allocated and cached: what one band
    at a time with twelve stored shortwave states took (2.6 GB measured; 4.2 with cotangents in arrays of their own)."""
    from rrtmgp_amd import _lib, device
    ncol, nlay, prec = 16384, 128, 4
    L = _lib.hip()

    def held():
        live, cached = C.c_size_t(0), C.c_size_t(0)
        _lib.check_hip(L.rrtmgp_hip_cache_stats(C.byref(live), C.byref(cached)))
        return live.value, cached.value

    atm = syn.make_atmosphere(syn.SEED_ATMOS[1], ncol, nlay, cloudy=True)
    kl, ks = G.KDist(kd_lw, AVAILABLE, prec), G.KDist(kd_sw, AVAILABLE, prec)
    sl, ss = G.SolverLW(kl, G.Cloud(lut_lw, prec)), G.SolverSW(ks, G.Cloud(lut_sw, prec))
    da = G.DeviceAtmosphere(atm, prec)
    c = device.DeviceArray.from_host(np.ones((ncol, nlay + 1)), np.float32)
    tsi = device.DeviceArray.from_host(np.ones(ncol), np.float32)
    device.synchronize()
    _lib.check_hip(L.rrtmgp_hip_cache_release())
    before = held()[0]
    sl.adjoint(da, c, c)
    ss.adjoint(da, tsi, c, c, c)
    device.synchronize()
    after = sum(held()) - before
    assert after <= 3.1e9, after


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("top_at_1", [0, 1])
def test_cotangents_over_inputs(G, precision, top_at_1):
    """Bit for bit what arrays of their own receive; 7 layers are one whole segment and part of another."""
    from rrtmgp_amd import _lib
    dt, suf = G.real_dtype(precision), "f64" if precision == 8 else "f32"
    ncol, nlay, nbnd, ng = 65, 7, 2, 21
    rng = np.random.default_rng(2)
    dev = lambda a: G.DeviceArray.from_host(np.asfortranarray(a), dt)          # noqa: E731
    u = lambda *s: rng.uniform(0.1, 0.9, s)                                     # noqa: E731
    i, full, lev = C.c_int64, (ncol, nlay, ng), (ncol, nlay + 1)
    head = [i(ncol), i(nlay), i(ng), C.c_int(top_at_1)]
    lims = np.array([1, 16, 17, 21], np.int32)
    lay, blev, emis, sfc, au, ad, ar = (dev(u(*s)) for s in ((ncol, nlay, nbnd), (ncol, nlay + 1, nbnd), (nbnd, ncol),
                                                             (ncol, ng), lev, lev, lev))
    tau, pf, ssa, g = u(*full), u(*full), u(*full), u(*full)
    mu0, alb, inc = dev(u(ncol)), dev(u(ncol, ng)), dev(u(ncol, ng))

    def lw(over):
        t, p = dev(tau), dev(pf)
        out = [t, p] if over else [G.DeviceArray(full, dt), G.DeviceArray(full, dt)]
        out += [G.DeviceArray((ncol, nlay, 2), dt) for _ in range(3)] + [G.DeviceArray((ncol, ng), dt) for _ in range(2)]
        _lib.check_hip(getattr(_lib.hip(), "rrtmgp_hip_lw_adjoint_factored_" + suf)(
            *head, C.c_double(1.66), C.c_double(0.5), t.ptr, p.ptr, lay.ptr, blev.ptr, i(nbnd),
            lims.ctypes.data_as(C.c_void_p), emis.ptr, i(nbnd), sfc.ptr, au.ptr, ad.ptr, *[o.ptr for o in out], None))
        return [_host(o) for o in out]

    def sw(over):
        t, w, a = dev(tau), dev(ssa), dev(g)
        out = [t, w] if over else [G.DeviceArray(full, dt), G.DeviceArray(full, dt)]
        out += [G.DeviceArray((ncol, ng), dt) for _ in range(2)]
        _lib.check_hip(getattr(_lib.hip(), "rrtmgp_hip_sw_adjoint_gases_" + suf)(
            *head, t.ptr, w.ptr, a.ptr, mu0.ptr, alb.ptr, alb.ptr, inc.ptr, None, au.ptr, ad.ptr, ar.ptr,
            *[o.ptr for o in out], None))
        return [_host(o) for o in out]

    for f in (lw, sw):
        for a, b in zip(f(False), f(True)):
            assert np.any(a != 0) and np.array_equal(a, b), f.__name__
