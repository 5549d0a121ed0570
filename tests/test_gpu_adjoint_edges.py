"""Shortwave solver adjoint at the edges of its layer formulas and tiles, against central differences
of the FP64 oracle, column by column.

Each column takes one (tau, ssa, g, mu0) regime in every layer: k mu0 within 1e-3 and 0.3 of 1 (the
removable singularity and both sides of its series), thin and thick layers, near-conservative and pure
absorption.  One layer, an odd few, and a second column tile with one column; 5 g-points fill one
work-group row and start another.

Bar: 1e-6 of sum |gradient x direction|.  The difference quotient (step h = 1e-5, relative) is off by
~h^2 = 1e-10 of it and by eps / h / |1 - k mu0| <= 2e-16 / 1e-5 / 1e-3 = 2e-8 from the oracle's rounding.
"""
import numpy as np
import pytest

from test_gpu_adjoint import G, _sw_adjoint   # noqa: F401  (G is a fixture)

pytestmark = pytest.mark.gpu


def _mu0_at(w0, g, kmu):
    g1, g2 = (8 - w0 * (5 + 3 * g)) / 4, 3 * w0 * (1 - g) / 4
    return kmu / np.sqrt((g1 - g2) * (g1 + g2))


@pytest.mark.parametrize("nlay,top_at_1", [(1, True), (2, False), (7, True)])
def test_sw_solver_adjoint_regimes(G, O, nlay, top_at_1):
    regimes = [(1.0, 0.3, 0.1, 1 + 1e-3), (1.0, 0.3, 0.1, 1 - 1e-3), (1e-3, 0.5, 0.0, 1 + 1e-3), (2.0, 0.4, 0.3, 0.7),
               (3.0, 0.2, 0.5, 1.3), (0.05, 0.6, 0.7, 0.8), (1e-6, 0.9, 0.0, 0.5), (30.0, 0.95, 0.8, 0.4),
               (5.0, 1 - 1e-6, 0.85, None), (0.2, 1e-9, 0.0, 0.9)]
    ncol, ngpt = 65, 5
    rng = np.random.default_rng(3)
    tau, ssa, g = (np.empty((ncol, nlay, ngpt)) for _ in range(3))
    mu0 = np.empty(ncol)
    for c in range(ncol):
        t, w, gg, kmu = regimes[c % len(regimes)]
        mu0[c] = 0.6 if kmu is None else min(_mu0_at(w, gg, kmu), 1.0)
        tau[c], ssa[c], g[c] = t * rng.uniform(0.99, 1.01, (nlay, ngpt)), w, gg
    bl = np.array([[1], [ngpt]], dtype=np.int32)
    alb = rng.uniform(0.1, 0.5, (1, ncol))
    toa = rng.uniform(1.0, 2.0, (ncol, ngpt))
    a_up, a_dn, a_dir = (rng.normal(size=(ncol, nlay + 1)) for _ in range(3))
    spread = lambda a: np.repeat(a.T, ngpt, axis=1)                        # noqa: E731
    grad = _sw_adjoint(G, tau, ssa, g, mu0, toa, spread(alb), spread(0.5 * alb), a_up, a_dn, a_dir, top_at_1, 8)

    def loss(x):
        up, dn, dr = O.rte_sw(x["tau"], x["ssa"], x["g"], mu0, toa, alb, 0.5 * alb, bl, top_at_1, do_broadband=True)
        return (a_up * up + a_dn * dn + a_dir * dr).sum(axis=1)

    base = {"tau": tau, "ssa": ssa, "g": g}
    h = 1e-5
    for name in base:
        size = {"tau": tau, "ssa": np.minimum(ssa, 1 - ssa), "g": np.minimum(g, 1 - g)}[name]
        v = rng.normal(size=tau.shape) * size
        fd = (loss({**base, name: base[name] + h * v}) - loss({**base, name: base[name] - h * v})) / (2 * h)
        ad = (grad[name] * v).sum(axis=(1, 2))
        scale = np.abs(grad[name] * v).sum(axis=(1, 2))
        # The oracle's own fluxes carry ~eps of their size, over h, into the quotient.
        noise = 4e-16 * np.abs(np.stack([a_up, a_dn, a_dir])).sum(axis=(0, 2)) * toa.sum(axis=1) / h
        bad = np.abs(ad - fd) > 1e-6 * scale + noise / 1e-3
        assert not bad.any(), (name, np.flatnonzero(bad)[:5], ad[bad][:5], fd[bad][:5])
