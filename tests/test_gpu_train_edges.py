"""Training gradients at batches that do and do not fill the kernels' 16-row groups, 32-row products and
row ranges (one row; a partial group; a partial product; several ranges with a short last one), for 512 and
448 outputs (the last 128-output pass half empty).

Reference: the network in FP64 with the kernels' BF16 rounding points.  A BF16 rounding that falls the other
way (its argument differs by FP32 rounding) moves one term by 2^-8; over n terms a gradient entry moves by at
most 2^-8 of its largest term, which the bound of 2^-7 of the array's largest entry covers for one row, and
random signs make it smaller for more.  In the 2-norm few entries are hit: 5e-3.
"""
import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_mlp import _np_forward, bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lw", [True, False])
@pytest.mark.parametrize("batch", [1, 17, 48, 100, 1056, 2500])
def test_gradients(syn, lw, batch):
    from rrtmgp_amd import api, surrogate as S
    from rrtmgp_amd.device import DeviceArray
    kd = api.KDist(syn.make_kdist(lw, 11 if lw else 12), AVAILABLE, precision=4)
    ts = S.build_training_set(kd, [syn.make_atmosphere(9, 64, 40)], seed=3)
    net = S.MlpGasOptics(kd, seed=5)
    net.fit_normalisation(ts)
    rng = np.random.default_rng(batch)
    for k, n in (("b1", 128), ("b2", 128), ("b3", net.n_out)):
        getattr(net, k).p = DeviceArray.from_host(rng.normal(0, 0.1, n).astype(np.float32), np.float32)
    idx = rng.integers(0, ts.rows, batch)
    w = net.host_weights()
    loss = net.forward_backward(ts, idx).to_host()
    got = {k: getattr(net, k).g.to_host().reshape(getattr(net, k).shape) for k in ("W1", "b1", "W2", "b2", "W3", "b3")}
    hs = {k: np.asarray(v, np.float32) for k, v in net.host_stats.items()}
    X, Y = ts.X.to_host().T[idx], ts.Y.to_host().T[idx]
    xn = np.zeros((batch, 16), np.float32)
    xn[:, :8] = (X[:, :8] - hs["x_mean"]) / hs["x_std"]
    xn = bf16(xn)
    yn = (Y - hs["y_mean"]) / hs["y_std"]
    z1, h1, z2, h2, y = _np_forward(w, xn)
    dy = 2.0 * (y - yn) / y.size
    np.testing.assert_allclose(loss.sum(dtype=np.float64) / y.size, np.mean((y - yn) ** 2), rtol=2e-3)
    dy16 = bf16(dy.astype(np.float32))
    dz2 = dy16 @ bf16(w["W3"]) / (1.0 + np.exp(-z2))
    dz2_16 = bf16(dz2.astype(np.float32))
    dz1 = dz2_16 @ bf16(w["W2"]) / (1.0 + np.exp(-z1))
    ref = {"W3": dy16.T @ h2, "b3": dy.sum(0), "W2": dz2_16.T @ h1, "b2": dz2.sum(0),
           "W1": bf16(dz1.astype(np.float32)).T @ xn, "b1": dz1.sum(0)}
    for k in ref:
        assert np.abs(got[k] - ref[k]).max() < 2.0 ** -7 * np.abs(ref[k]).max(), k
        assert np.linalg.norm(got[k] - ref[k]) < 5e-3 * np.linalg.norm(ref[k]), k
    again = net.forward_backward(ts, idx).to_host()
    assert np.array_equal(again, loss)
    for k in got:
        assert np.array_equal(getattr(net, k).g.to_host().reshape(got[k].shape), got[k]), k


def test_adam_arrays(syn):
    """One launch over all parameters against the recurrence in FP32 numpy."""
    from rrtmgp_amd import api, surrogate as S
    from rrtmgp_amd.device import DeviceArray
    kd = api.KDist(syn.make_kdist(False, 12), AVAILABLE, precision=4)
    net = S.MlpGasOptics(kd, seed=5)
    rng = np.random.default_rng(1)
    before = []
    for p in net.params:
        p.g = DeviceArray.from_host(rng.normal(0, 1, p.n).astype(np.float32), np.float32)
        before.append((p.p.to_host(), p.g.to_host()))
    net.adam_step(1e-3)
    for p, (p0, g) in zip(net.params, before):
        np.testing.assert_allclose(p.m.to_host(), 0.1 * g, rtol=1e-5)
        np.testing.assert_allclose(p.v.to_host(), 1e-3 * g * g, rtol=1e-4)
        # First step: m / c1 = g, v / c2 = g^2, so each weight moves by lr against its gradient's sign.
        np.testing.assert_allclose(p.p.to_host() - p0, -1e-3 * np.sign(g), rtol=2e-3, atol=3e-7)
        if p.b16 is not None:
            b = p.b16.to_host().astype(np.uint32) << 16
            assert np.array_equal(b.view(np.float32), bf16(p.p.to_host()).astype(np.float32))
