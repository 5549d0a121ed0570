"""Device-array pool: reuse rules on the host, and calls whose outputs land in reused memory."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import AVAILABLE

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool_policy(tmp_path):
    src = os.path.join(ROOT, "tests", "native", "device_pool_check.cpp")
    exe = str(tmp_path / "device_pool_check")
    inc = os.path.join(ROOT, "rte-rrtmgp-cpp_amd", "csrc")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", inc, src, "-o", exe],
                       capture_output=True, text=True)
    if r.returncode != 0:
        pytest.fail(r.stderr)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.strip() == "ok"


def _poison(shapes, dt):
    """Leaves freed blocks of these sizes, all bytes set (NaN in floating point), in the pool."""
    from rrtmgp_amd import _lib
    from rrtmgp_amd.device import DeviceArray
    held = [DeviceArray(s, dt, zero=False) for s in shapes for _ in range(8)]
    for a in held:
        _lib.check_hip(_lib.hip().rrtmgp_hip_memset(a.ptr, 255, C.c_size_t(a.nbytes), None))


@pytest.mark.gpu
@pytest.mark.parametrize("precision,ncol,nlay", [(8, 1, 1), (4, 65, 7), (8, 130, 10)])
def test_outputs_in_reused_memory(precision, ncol, nlay):
    """Every element of every output is written: results do not depend on what the memory held."""
    from rrtmgp_amd import api, synthetic
    dt = api.real_dtype(precision)
    kl = api.KDist(synthetic.make_kdist(True, 11), AVAILABLE, precision)
    ks = api.KDist(synthetic.make_kdist(False, 12), AVAILABLE, precision)
    atm = synthetic.make_atmosphere(4, ncol, nlay)
    shapes = [(ncol, nlay), (ncol, nlay + 1)]
    shapes += [s + (n,) for s in shapes for n in (kl.nbnd, ks.nbnd, kl.ngpt, ks.ngpt, kl.ngas)]
    shapes += [(ncol, n) for n in (kl.ngpt, ks.ngpt, kl.nbnd, ks.nbnd)] + [(ncol,)]

    def run():
        got = {}
        gas = api.GasConcs(atm.vmr, precision)
        cd = api.get_col_dry(atm.vmr["h2o"], atm.p_lev, precision)
        got["col_dry"] = cd
        lw = api.gas_optics(kl, atm, gas, cd)
        sw = api.gas_optics(ks, atm, gas, cd)
        got.update({"lw_" + k: v for k, v in lw.items()})
        got.update({"sw_" + k: v for k, v in sw.items()})
        for bb in (False, True):
            u, d = api.rte_lw(kl, False, lw["tau"], lw["lay_src"], lw["lev_src_inc"], lw["lev_src_dec"],
                              lw["sfc_src"], atm.emis_sfc, do_broadband=bb)
            got.update({f"lw_up{bb}": u, f"lw_dn{bb}": d})
            if not bb:
                got.update({"red_" + k: v for k, v in api.fluxes_reduce(kl, u, d, byband=True).items()})
            us, ds, rs = api.rte_sw(ks, False, sw["tau"], sw["ssa"], sw["g"], atm.mu0, sw["toa_src"],
                                    atm.sfc_alb, atm.sfc_alb, do_broadband=bb)
            got.update({f"sw_up{bb}": us, f"sw_dn{bb}": ds, f"sw_dir{bb}": rs})
        o = api.rte_sw_bnd(ks, False, sw["tau"], sw["ssa"], sw["g"], atm.mu0, sw["toa_src"], atm.sfc_alb,
                           atm.sfc_alb, p_lev=atm.p_lev)
        got.update({"bnd_" + k: v for k, v in o.items()})
        got["hr"] = api.heating_rate(o["flux_up"], o["flux_dn"], atm.p_lev, precision)
        da = api.DeviceAtmosphere(atm, precision)
        sl, ss = api.SolverLW(kl), api.SolverSW(ks)
        tsi = np.ones(ncol)
        got.update({"sl_" + k: v for k, v in sl.solve(da, bnd=True, heating_rate=True).items() if v is not None})
        got.update({"ss_" + k: v for k, v in ss.solve(da, tsi, bnd=True, heating_rate=True).items()
                    if v is not None})
        c = np.ones((ncol, nlay + 1))
        got.update({"al_" + k: v for k, v in sl.adjoint(da, c, c).items()})
        got.update({"as_" + k: v for k, v in ss.adjoint(da, tsi, c, c, c).items()})
        return {k: v.to_host() for k, v in got.items()}

    fresh = run()
    _poison(shapes, dt)
    again = run()
    assert fresh.keys() == again.keys() and len(fresh) > 50
    for k in fresh:
        assert np.isfinite(again[k]).all(), k
        np.testing.assert_allclose(again[k], fresh[k], rtol=1e-5 if precision == 4 else 1e-11,
                                   atol=1e-5 * np.abs(fresh[k]).max(initial=0.0), err_msg=k)


@pytest.mark.gpu
def test_held_blocks_go_back_when_memory_runs_out():
    """What the pool holds is there for the library's other allocations: with 6 GiB of the device left, 4 of them
    freed into the pool, another 5 GiB are found through each entry.  Nothing touches the memory."""
    torch = pytest.importorskip("torch")
    from rrtmgp_amd import _lib
    L, gib = _lib.hip(), 1 << 30
    new = lambda entry, n, *a: (lambda p: (getattr(L, entry)(C.byref(p), C.c_size_t(n), *a), p))(C.c_void_p())   # noqa: E731
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    _lib.check_hip(L.rrtmgp_hip_cache_release())
    rc, rest = new("rrtmgp_hip_malloc", torch.cuda.mem_get_info()[0] - 6 * gib)
    assert rc == 0
    try:
        for entry, drop in (("rrtmgp_hip_malloc", L.rrtmgp_hip_free), ("rrtmgp_hip_pool_malloc", L.rrtmgp_hip_pool_free),
                            ("rrtmgp_hip_cache_malloc", lambda p: L.rrtmgp_hip_cache_free(p, None))):
            rc, p = new("rrtmgp_hip_pool_malloc", 4 * gib)
            assert rc == 0 and L.rrtmgp_hip_pool_free(p) == 0
            rc, p = new(entry, 5 * gib, *([None] if "cache" in entry else []))
            assert rc == 0, entry
            assert drop(p) == 0
            _lib.check_hip(L.rrtmgp_hip_cache_release())
    finally:
        L.rrtmgp_hip_free(rest)


@pytest.mark.gpu
def test_stats():
    import gc
    from rrtmgp_amd import _lib
    from rrtmgp_amd.device import DeviceArray
    L = _lib.hip()

    def stats():
        live, held = C.c_size_t(0), C.c_size_t(0)
        _lib.check_hip(L.rrtmgp_hip_pool_stats(C.byref(live), C.byref(held)))
        return np.array([live.value, held.value], dtype=np.int64)

    gc.collect()                                       # arrays that earlier tests left in reference cycles
    _lib.check_hip(L.rrtmgp_hip_cache_release())
    before, mib = stats(), 1 << 20
    assert before[1] == 0
    a = [DeviceArray((n,), np.uint8, zero=False) for n in (4 * mib, 1000)]
    assert list(stats() - before) == [4 * mib + 1024, 0]
    a[0].free()
    assert list(stats() - before) == [1024, 4 * mib]
    a[1].free()
    assert list(stats() - before) == [0, 4 * mib + 1024]
    _lib.check_hip(L.rrtmgp_hip_cache_release())
    assert list(stats() - before) == [0, 0]
