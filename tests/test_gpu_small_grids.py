"""Calls too small to fill the chip cut the bands over more work-groups (solvers: 8 or 4 g-points each; gas
optics: fewer bands each).  The same columns as part of a call that is not cut give the same bits; column
counts around the tile and split edges, with the ragged bands (1 to 33 g-points) of the gas-optics tests.
"""
import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_adjoint import G, _host                           # noqa: F401  (G is a fixture)
from test_gpu_gas_optics_adjoint import ragged

pytestmark = pytest.mark.gpu

BIG = 64 * 64                   # 64 tiles x 9 groups: not cut


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("ncol", [1, 63, 65, 257, 600, 1100])
def test_split_matches_whole(G, syn, precision, ncol):
    from dataclasses import replace
    nlay = 11
    big = syn.make_atmosphere(4, BIG, nlay, cloudy=True)
    nb = {True: 6, False: 6}
    big = replace(big, emis_sfc=np.asfortranarray(big.emis_sfc[:nb[True]]),
                  sfc_alb=np.asfortranarray(big.sfc_alb[:nb[False]]))
    small = syn.subset_columns(big, np.arange(ncol))
    kl = G.KDist(ragged(syn.make_kdist(True, 11)), AVAILABLE, precision)
    ks = G.KDist(ragged(syn.make_kdist(False, 12)), AVAILABLE, precision)

    def run(atm):
        n = atm.p_lay.shape[0]
        da = G.DeviceAtmosphere(atm, precision, cloudy=False)
        out = {}
        for lw, k in ((True, kl), (False, ks)):
            cd = G.get_col_dry(atm.vmr["h2o"], atm.p_lev, precision)
            out.update({f"gas {lw} {m}": _host(v) for m, v in G.gas_optics(k, da, da.gas_concs, cd).items()})
        out.update({"lw " + m: _host(v) for m, v in
                    G.SolverLW(kl).solve(da, bnd=True, heating_rate=True).items() if v is not None})
        out.update({"sw " + m: _host(v) for m, v in
                    G.SolverSW(ks).solve(da, np.ones(n), bnd=True, heating_rate=True).items() if v is not None})
        return out

    whole, part = run(big), run(small)
    assert whole.keys() == part.keys()
    for k in whole:
        assert np.array_equal(part[k], whole[k][:ncol]), k


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("ncol", [1, 65, 600])
def test_split_matches_whole_every_form(G, syn, precision, ncol):
    """The same for every variant of the solver kernels: drivers with and without heating rates and band fluxes
    (factored sources, co-albedo), and the class calls (separate sources, 1 to 4 angles, single-scattering
    albedo or co-albedo; broadband and g-point fluxes, band fluxes with heating rates)."""
    from dataclasses import replace
    nlay = 11
    big = syn.make_atmosphere(4, BIG, nlay)
    big = replace(big, emis_sfc=np.asfortranarray(0.9 * big.emis_sfc[:6]), sfc_alb=np.asfortranarray(big.sfc_alb[:6]))
    small = syn.subset_columns(big, np.arange(ncol))
    kl = G.KDist(ragged(syn.make_kdist(True, 11)), AVAILABLE, precision)
    ks = G.KDist(ragged(syn.make_kdist(False, 12)), AVAILABLE, precision)

    def run(atm):
        n = atm.p_lay.shape[0]
        da = G.DeviceAtmosphere(atm, precision, cloudy=False)
        cd = G.get_col_dry(atm.vmr["h2o"], atm.p_lev, precision)
        out = {}
        for hr in (False, True):
            for bnd in (False, True):
                o = {"lw": G.SolverLW(kl).solve(da, bnd=bnd, heating_rate=hr),
                     "sw": G.SolverSW(ks).solve(da, np.ones(n), bnd=bnd, heating_rate=hr)}
                out.update({f"{r} {hr} {bnd} {m}": v for r, f in o.items() for m, v in f.items() if v is not None})
        a = G.gas_optics(kl, da, da.gas_concs, cd)
        for bb in (False, True):
            for mu in (1, 2, 3, 4):
                o = G.rte_lw(kl, False, a["tau"], a["lay_src"], a["lev_src_inc"], a["lev_src_dec"], a["sfc_src"],
                             atm.emis_sfc, n_gauss_angles=mu, do_broadband=bb)
                out.update({f"rte_lw {bb} {mu} {i}": v for i, v in enumerate(o)})
        for co in (False, True):
            b = G.gas_optics(ks, da, da.gas_concs, cd, coalbedo=co)
            w = b["coalbedo" if co else "ssa"]
            if not co:
                for bb in (False, True):
                    o = G.rte_sw(ks, False, b["tau"], w, b["g"], atm.mu0, b["toa_src"], atm.sfc_alb, atm.sfc_alb,
                                 do_broadband=bb)
                    out.update({f"rte_sw {bb} {i}": v for i, v in enumerate(o)})
            for p in (None, atm.p_lev):
                o = G.rte_sw_bnd(ks, False, b["tau"], w, b["g"], atm.mu0, b["toa_src"], atm.sfc_alb, atm.sfc_alb,
                                 p_lev=p, coalbedo=co)
                out.update({f"rte_sw_bnd {co} {p is None} {m}": v for m, v in o.items() if v is not None})
        return {k: _host(v) for k, v in out.items()}

    whole, part = run(big), run(small)
    assert whole.keys() == part.keys()
    bad = [k for k in whole if not np.array_equal(part[k], whole[k][:ncol])]
    assert not bad, bad
