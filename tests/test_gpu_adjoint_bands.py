"""The adjoint drivers on more bands than one launch of the longwave solver adjoint takes (258 of one g-point)."""
import copy

import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_adjoint import G, _directions, _dot, _host, _perturbed   # noqa: F401  (G is a fixture)

pytestmark = pytest.mark.gpu

NB = 258


def many_bands(kd):
    """NB bands of one g-point each, taken in turn from the bands of a synthetic k-distribution."""
    nb0 = kd.nbnd
    src, gpt = np.arange(NB) % nb0, np.arange(NB) // nb0 % 16
    pick = 16 * src + gpt
    k = copy.deepcopy(kd)
    k.band2gpt = np.asfortranarray(np.tile(np.arange(1, NB + 1), (2, 1)).astype(np.int32))
    k.key_species = np.asfortranarray(kd.key_species[:, :, src])
    k.band_lims_wavenum = np.asfortranarray(kd.band_lims_wavenum[:, src])
    k.kmajor = np.asfortranarray(kd.kmajor[pick])
    for s in ("lower", "upper"):
        lim, start = getattr(kd, f"minor_limits_gpt_{s}"), getattr(kd, f"kminor_start_{s}")
        use = [(m, i) for i in range(NB) for m in range(lim.shape[1]) if (lim[0, m] - 1) // 16 == src[i]]
        ms = [m for m, _ in use]
        setattr(k, f"kminor_{s}", np.asfortranarray(getattr(kd, f"kminor_{s}")[[start[m] - 1 + gpt[i] for m, i in use]]))
        setattr(k, f"minor_limits_gpt_{s}", np.asfortranarray(np.array([[i + 1, i + 1] for _, i in use], np.int32).T))
        setattr(k, f"kminor_start_{s}", np.arange(1, len(use) + 1, dtype=np.int32))
        for f in ("minor_gases", "scaling_gas"):
            setattr(k, f"{f}_{s}", [getattr(kd, f"{f}_{s}")[m] for m in ms])
        for f in ("minor_scales_with_density", "scale_by_complement"):
            setattr(k, f"{f}_{s}", getattr(kd, f"{f}_{s}")[ms])
    if kd.is_lw:
        k.totplnk = np.asfortranarray(kd.totplnk[:, src])
        k.planck_frac = np.asfortranarray(kd.planck_frac[pick])
    else:
        for f in ("solar_src_quiet", "solar_src_facular", "solar_src_sunspot", "rayl_lower", "rayl_upper"):
            setattr(k, f, np.asfortranarray(getattr(kd, f)[pick]))
    return k


@pytest.mark.parametrize("lw", [True, False])
def test_many_bands(G, O, syn, kd_lw, kd_sw, lw):
    """End to end against the oracle (1e-5, as the other end-to-end tests)."""
    k = many_bands(kd_lw if lw else kd_sw)
    atm = syn.make_atmosphere(53, 3, 12, nbnd_lw=NB, nbnd_sw=NB)
    kd, okd = G.KDist(k, AVAILABLE, 8), O.Kdist(k, AVAILABLE)
    rng = np.random.default_rng(13)
    a = [rng.normal(size=(atm.ncol, atm.nlay + 1)) for _ in range(2 if lw else 3)]
    da = G.DeviceAtmosphere(atm, 8)
    if lw:
        grad = G.SolverLW(kd).adjoint(da, *a)
    else:
        tsi = np.full(atm.ncol, atm.tsi / kd.scalar("tsi"))
        grad = G.SolverSW(kd).adjoint(da, tsi, *a)
    grad = {n: _host(d) for n, d in grad.items()}

    def loss(at):
        o = O.solve_lw(okd, at) if lw else O.solve_sw(okd, at, tsi_scaling=tsi)
        return float(sum(np.sum(q * o[n]) for q, n in zip(a, ("flux_up", "flux_dn", "flux_dn_dir"))))

    v = _directions(rng, atm, lw)
    h = 1e-4
    fd = (loss(_perturbed(atm, v, h)) - loss(_perturbed(atm, v, -h))) / (2 * h)
    ad = _dot(G, grad, v, kd.gas_names, lw)
    assert abs(ad - fd) <= 1e-5 * abs(fd), (ad, fd)
