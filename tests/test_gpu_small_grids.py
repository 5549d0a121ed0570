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
