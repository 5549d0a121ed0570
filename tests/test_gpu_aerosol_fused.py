"""Aerosols added while the gas optics writes give what a separate add_to gives: the shortwave driver against
gas optics, cloud add_to, aerosol add_to and the solver called one by one, in the co-albedo form, for ragged
bands and column counts around the 64-column tile.

Both evaluate the same expressions; the compiler may contract a product and a sum in one and not in the
other, so the optical properties agree to a few eps and the fluxes, whose sensitivity to them is of order one
except near k mu0 = 1, to 1e-11 (FP64) and 1e-5 (FP32) of the largest flux.
"""
import os

import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_adjoint import G, _host                           # noqa: F401  (G is a fixture)
from test_gpu_aerosol import GOLD, _aerosols

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("ncol,nlay,cloudy", [(1, 3, True), (65, 12, True), (65, 12, False), (130, 5, True)])
def test_driver_matches_steps(G, syn, kd_sw, lut_sw, precision, ncol, nlay, cloudy):
    from rrtmgp_amd import coefficients, netcdf
    lut = coefficients.aerosol_lut(netcdf.Dataset(os.path.join(GOLD, "aerosol_optics.nc")))
    atm = syn.make_atmosphere(5, ncol, nlay, cloudy=True)
    kd = G.KDist(kd_sw, AVAILABLE, precision)
    cloud, aero = G.Cloud(lut_sw, precision), G.Aerosol(lut, precision)
    f, rh = _aerosols(ncol, nlay, 3)
    concs = G.GasConcs(f, precision)
    da = G.DeviceAtmosphere(atm, precision, cloudy=cloudy)
    got = G.SolverSW(kd, cloud, aero).solve(da, np.ones(ncol), aerosol=(rh, concs), heating_rate=True)
    o = G.gas_optics(kd, da, da.gas_concs, G.get_col_dry(atm.vmr["h2o"], atm.p_lev, precision), coalbedo=True)
    if cloudy:
        t, c, g = cloud.optics(atm.lwp, atm.iwp, atm.rel, atm.rei, True, delta_scale=True, coalbedo=True)
        G.add_to(kd, o["tau"], t, o["coalbedo"], o["g"], c, g, coalbedo=True)
    t, c, g = aero.optics(concs, rh, atm.p_lev, coalbedo=True)
    G.add_to(kd, o["tau"], t, o["coalbedo"], o["g"], c, g, coalbedo=True)
    want = G.rte_sw_bnd(kd, atm.top_at_1, o["tau"], o["coalbedo"], o["g"], atm.mu0, o["toa_src"], atm.sfc_alb,
                        atm.sfc_alb, p_lev=atm.p_lev, coalbedo=True)
    for k in ("flux_up", "flux_dn", "flux_dn_dir", "heating_rate"):
        a, b = _host(got[k]), _host(want[k])
        assert np.abs(a - b).max() <= (1e-5 if precision == 4 else 1e-11) * np.abs(b).max(), k
