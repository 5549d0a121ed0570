"""Shortwave solver adjoint at the edges of its layer formulas and tiles, column by column, against central
differences of the forward in 80-bit arithmetic (numpy's long double), which is itself held to the FP64 oracle.

Each column takes one (tau, ssa, g, mu0) regime in every layer: k mu0 within 1e-3 and 0.3 of 1 (the
removable singularity and both sides of its series), thin and thick layers, near-conservative and pure
absorption.  One layer, an odd few, and a second column tile with one column; 5 g-points fill one
work-group row and start another.

Bar: 1e-6 of sum |gradient x direction|, for every input and column.  Directions have the size of what is varied
(the distance to the bound for ssa, 0.1 for g = 0) and the step is 1e-4 of them, which leaves ~1e-8 of truncation;
3e-6 for the thick layers' tau, whose exponentials change by tau; and longer where the fluxes are linear in the
variation (ssa and g of thin or hardly scattering layers) or it is small against its scale (1 - ssa = 1e-6), so
that what rounding of the fluxes (~1e-19 / |1 - k mu0| of their sum) puts into the quotient, which is added to
the bar, is at most 2e-6 of the same sum.
"""
import numpy as np
import pytest

from test_gpu_adjoint import G, _sw_adjoint   # noqa: F401  (G is a fixture)

pytestmark = pytest.mark.gpu


def _mu0_at(w0, g, kmu):
    g1, g2 = (8 - w0 * (5 + 3 * g)) / 4, 3 * w0 * (1 - g) / 4
    return kmu / np.sqrt((g1 - g2) * (g1 + g2))


def _fluxes(tau, ssa, g, mu0, toa, alb_dir, alb_dif, top_at_1):
    """Broadband up, total down and direct fluxes (ncol, nlay + 1) by two-stream and adding, in long double."""
    E = np.longdouble
    if not top_at_1:
        tau, ssa, g = tau[:, ::-1], ssa[:, ::-1], g[:, ::-1]
    n, mu, eps = tau.shape[1], mu0.astype(E)[:, None], E(np.finfo(np.float64).eps)
    t, w, g = (np.moveaxis(x.astype(E), 1, 0) for x in (tau, ssa, g))
    g1, g2, g3 = (8 - w * (5 + 3 * g)) / 4, 3 * w * (1 - g) / 4, (2 - 3 * mu * g) / 4
    g4 = 1 - g3
    a1, a2 = g1 * g4 + g2 * g3, g1 * g3 + g2 * g4
    k = np.sqrt(np.maximum((g1 - g2) * (g1 + g2), E(1e-12)))
    e1 = np.exp(-t * k)
    e2, Tn, km = e1 * e1, np.exp(-t / mu), k * mu
    RT = 1 / (k * (1 + e2) + g1 * (1 - e2))
    R, T = RT * g2 * (1 - e2), RT * 2 * k * e1
    q = w * RT / (1 - km * km)
    Rd = q * ((1 - km) * (a2 + k * g3) - (1 + km) * (a2 - k * g3) * e2 - 2 * (k * g3 - a2 * km) * e1 * Tn)
    Td = -q * ((1 + km) * (a1 + k * g4) * Tn - (1 - km) * (a1 - k * g4) * e2 * Tn - 2 * (k * g4 + a1 * km) * e1)
    Rd = np.maximum(np.minimum(Rd, 1 - Tn), eps)
    Td = np.maximum(np.minimum(Td, 1 - Tn - Rd), eps)
    dir_ = [toa.astype(E) * mu]
    for j in range(n):
        dir_.append(dir_[j] * Tn[j])
    A, S = [alb_dif.astype(E)], [alb_dir.astype(E) * dir_[n]]          # below each level, from the surface up
    for j in range(n - 1, -1, -1):
        e = 1 / (1 - R[j] * A[0])
        S.insert(0, Rd[j] * dir_[j] + T[j] * (S[0] + A[0] * Td[j] * dir_[j]) * e)
        A.insert(0, R[j] + T[j] * T[j] * A[0] * e)
    dn = [np.zeros_like(dir_[0])]
    for j in range(n):
        dn.append((T[j] * dn[j] + R[j] * S[j + 1] + Td[j] * dir_[j]) / (1 - R[j] * A[j + 1]))
    out = [np.stack([x.sum(axis=-1) for x in f], axis=1) for f in
           ([A[j] * dn[j] + S[j] for j in range(n + 1)], [dn[j] + dir_[j] for j in range(n + 1)], dir_)]
    return out if top_at_1 else [x[:, ::-1] for x in out]


@pytest.mark.parametrize("nlay,top_at_1", [(1, True), (2, False), (7, True)])
def test_sw_solver_adjoint_regimes(G, O, nlay, top_at_1):
    regimes = [(1.0, 0.3, 0.1, 1 + 1e-3), (1.0, 0.3, 0.1, 1 - 1e-3), (1e-3, 0.5, 0.0, 1 + 1e-3), (2.0, 0.4, 0.3, 0.7),
               (3.0, 0.2, 0.5, 1.3), (0.05, 0.6, 0.7, 0.8), (1e-6, 0.9, 0.0, 0.5), (30.0, 0.95, 0.8, 0.4),
               (5.0, 1 - 1e-6, 0.85, None), (0.2, 1e-9, 0.0, 0.9)]
    steps = {"tau": [1e-4] * 7 + [3e-6, 1e-4, 1e-4], "ssa": [1e-4] * 6 + [1e-3, 1e-4, 1e-2, 0.1],
             "g": [1e-4, 1e-4, 1e-3, 1e-4, 1e-4, 1e-4, 1e-2, 1e-4, 1e-4, 3.0]}
    ncol, ngpt = 65, 5
    off = np.array([1e-3 if r[3] is not None and abs(r[3] - 1) < 0.01 else 1.0 for r in regimes])[np.arange(ncol) % len(regimes)]
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

    def fluxes(x):
        return _fluxes(x["tau"], x["ssa"], x["g"], mu0, toa, spread(alb), spread(0.5 * alb), top_at_1)

    def loss(x):
        up, dn, dr = fluxes(x)
        return (a_up * up + a_dn * dn + a_dir * dr).sum(axis=1)

    base = {"tau": tau, "ssa": ssa, "g": g}
    for x, y in zip(fluxes(base), O.rte_sw(tau, ssa, g, mu0, toa, alb, 0.5 * alb, bl, top_at_1, do_broadband=True)):
        np.testing.assert_allclose(x.astype(np.float64), y, rtol=1e-11, atol=1e-12)     # oracle: ~eps / |1 - k mu0|
    for name in base:
        size = {"tau": tau, "ssa": np.minimum(ssa, 1 - ssa), "g": np.where(g == 0, 0.1, np.minimum(g, 1 - g))}[name]
        v = rng.normal(size=tau.shape) * size
        h = np.array(steps[name])[np.arange(ncol) % len(regimes)]
        x = {s: {**base, name: base[name].astype(np.longdouble) + s * h[:, None, None] * v} for s in (1, -1)}
        fd = (loss(x[1]) - loss(x[-1])) / (2 * h)
        ad = (grad[name] * v).sum(axis=(1, 2))
        scale = np.abs(grad[name] * v).sum(axis=(1, 2))
        total = np.abs(np.stack([a_up, a_dn, a_dir])).sum(axis=(0, 2)) * toa.sum(axis=1)
        noise = np.finfo(np.longdouble).eps * total / h / off
        assert (noise <= 2e-6 * scale).all(), name          # every column counts
        bad = np.abs(ad - fd) > 1e-6 * scale + noise
        assert not bad.any(), (name, np.flatnonzero(bad)[:5], ad[bad][:5], fd[bad][:5], (np.abs(ad - fd) / scale).max())
