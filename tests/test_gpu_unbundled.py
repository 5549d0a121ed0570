"""Kernel entry points whose work the library's own paths do in fused kernels: the training building blocks, put
together to one step, and the separate flux sums, each against the fused form."""
import ctypes as C

import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_adjoint import G, _host                           # noqa: F401  (G is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lw,batch", [(True, 100), (False, 1056)])
def test_training_step(syn, lw, batch):
    """Both forms round to BF16 at the same points and differ in the order of FP32 sums, which turns a BF16
    rounding over (2^-8 of one term) now and then: 5e-3 in the 2-norm of each gradient, as in the tests of the
    fused step.  Adam's arithmetic is the same: bit for bit from the same gradients."""
    from rrtmgp_amd import _lib, api, surrogate as S
    from rrtmgp_amd.device import DeviceArray
    L, i, f, h = _lib.hip(), C.c_int64, C.c_float, 128
    chk = _lib.check_hip
    kd = api.KDist(syn.make_kdist(lw, 11 if lw else 12), AVAILABLE, precision=4)
    ts = S.build_training_set(kd, [syn.make_atmosphere(9, 64, 40)], seed=3)
    net = S.MlpGasOptics(kd, seed=5)
    net.fit_normalisation(ts)
    rng = np.random.default_rng(batch)
    for k, n in (("b1", h), ("b2", h), ("b3", net.n_out)):
        getattr(net, k).p = DeviceArray.from_host(rng.normal(0, 0.1, n).astype(np.float32), np.float32)
    rows = rng.integers(0, ts.rows, batch)
    loss = net.forward_backward(ts, rows).to_host().sum(dtype=np.float64)
    names = ("W1", "b1", "W2", "b2", "W3", "b3")
    fused = {k: getattr(net, k).g.to_host().astype(np.float64) for k in names}

    no, st = net.n_out, net.stats
    f32 = lambda *s: DeviceArray(s, np.float32)                         # noqa: E731
    b16 = lambda *s: DeviceArray(s, np.uint16)                          # noqa: E731
    idx = DeviceArray.from_host(rows.astype(np.int64), np.int64)
    xr, yr, x16, yn = f32(batch * 16), f32(batch * no), b16(batch * 16), f32(batch * no)
    z1, h1, z2, h2, y = f32(batch * h), b16(batch * h), f32(batch * h), b16(batch * h), f32(batch * no)
    dy16, dyf, parts = b16(batch * no), f32(batch * no), f32((batch * no + 255) // 256)
    dh, dz16, dzf = f32(batch * h), b16(batch * h), f32(batch * h)
    g = {k: f32(getattr(net, k).n) for k in names}

    def gemm(M, N, K, A, sAm, sAk, B, sBk, sBn, out, sCm, sCn):
        chk(L.rrtmgp_hip_mlp_gemm_bf16(i(M), i(N), i(K), A.ptr, i(sAm), i(sAk), B.ptr, i(sBk), i(sBn), out.ptr,
                                       i(sCm), i(sCn), C.c_int(0), None))

    B = batch
    for n, n_norm, src, raw, mean, std, o16, o32 in ((16, 8, ts.X, xr, "x_mean", "x_std", x16.ptr, None),
                                                     (no, no, ts.Y, yr, "y_mean", "y_std", None, yn.ptr)):
        chk(L.rrtmgp_hip_mlp_gather_rows(i(B), C.c_int(n), idx.ptr, src.ptr, raw.ptr, None))
        chk(L.rrtmgp_hip_mlp_normalize_rows(i(B), C.c_int(n), C.c_int(n_norm), raw.ptr, st[mean].ptr, st[std].ptr,
                                            o16, o32, None))
    for x, n_in, w, b, z, out in ((x16, 16, net.W1, net.b1, z1, h1), (h1, h, net.W2, net.b2, z2, h2)):
        gemm(B, h, n_in, x, n_in, 1, w.b16, 1, n_in, z, h, 1)
        chk(L.rrtmgp_hip_mlp_bias_softplus(i(B), C.c_int(h), z.ptr, b.p.ptr, out.ptr, None))
    gemm(B, no, h, h2, h, 1, net.W3.b16, 1, h, y, no, 1)
    chk(L.rrtmgp_hip_mlp_mse_grad(i(B), C.c_int(no), y.ptr, net.b3.p.ptr, yn.ptr, dy16.ptr, dyf.ptr, parts.ptr, None))
    gemm(no, h, B, dy16, 1, no, h2, h, 1, g["W3"], h, 1)
    chk(L.rrtmgp_hip_mlp_bias_grad(i(B), C.c_int(no), dyf.ptr, g["b3"].ptr, None))
    gemm(B, h, no, dy16, no, 1, net.W3.b16, h, 1, dh, h, 1)
    chk(L.rrtmgp_hip_mlp_softplus_back(i(B * h), dh.ptr, z2.ptr, dz16.ptr, dzf.ptr, None))
    gemm(h, h, B, dz16, 1, h, h1, h, 1, g["W2"], h, 1)
    chk(L.rrtmgp_hip_mlp_bias_grad(i(B), C.c_int(h), dzf.ptr, g["b2"].ptr, None))
    gemm(B, h, h, dz16, h, 1, net.W2.b16, h, 1, dh, h, 1)
    chk(L.rrtmgp_hip_mlp_softplus_back(i(B * h), dh.ptr, z1.ptr, dz16.ptr, dzf.ptr, None))
    gemm(h, 16, B, dz16, 1, h, x16, 16, 1, g["W1"], 16, 1)
    chk(L.rrtmgp_hip_mlp_bias_grad(i(B), C.c_int(h), dzf.ptr, g["b1"].ptr, None))
    np.testing.assert_allclose(parts.to_host().sum(dtype=np.float64), loss, rtol=1e-3)
    for k in names:
        assert np.linalg.norm(g[k].to_host() - fused[k]) < 5e-3 * np.linalg.norm(fused[k]), k

    # Adam on one array at a time and on all at once, twice, from the same state.
    copy = lambda a: DeviceArray.from_host(a.to_host(), a.dtype)        # noqa: E731
    own = [{m: copy(getattr(p, m)) for m in ("p", "g", "m", "v")} | {"b16": copy(p.b16) if p.b16 is not None else None}
           for p in net.params]
    for step in (1, 2):
        net.adam_step(1e-3)
        for p, o in zip(net.params, own):
            chk(L.rrtmgp_hip_mlp_adam(i(p.n), o["p"].ptr, o["g"].ptr, o["m"].ptr, o["v"].ptr,
                                      o["b16"].ptr if o["b16"] is not None else None, f(1e-3), f(0.9), f(0.999), f(1e-8),
                                      i(step), None))
    for p, o in zip(net.params, own):
        for m in ("p", "m", "v", "b16"):
            if o[m] is not None:
                assert np.array_equal(o[m].to_host(), getattr(p, m).to_host()), m


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("ncol,nlev,ngpt", [(1, 1, 1), (65, 7, 37), (257, 3, 64)])
def test_flux_sums(G, precision, ncol, nlev, ngpt):
    """Sums in g-point order in the build's precision, bit for bit those of the fused reduction."""
    from rrtmgp_amd import _lib
    dt, suf = G.real_dtype(precision), "f64" if precision == 8 else "f32"
    L, i = _lib.hip(), C.c_int64
    rng = np.random.default_rng(ngpt)
    up, dn = (G.DeviceArray.from_host(rng.uniform(0, 10, (ncol, nlev, ngpt)), dt) for _ in range(2))
    one, all_ = ([G.DeviceArray((ncol, nlev), dt) for _ in range(3)] for _ in range(2))
    for src, out in ((up, one[0]), (dn, one[1])):
        _lib.check_hip(getattr(L, "rrtmgp_hip_sum_broadband_" + suf)(i(ncol), i(nlev), i(ngpt), src.ptr, out.ptr, None))
    _lib.check_hip(getattr(L, "rrtmgp_hip_net_broadband_" + suf)(i(ncol), i(nlev), one[1].ptr, one[0].ptr, one[2].ptr,
                                                                 None))
    _lib.check_hip(getattr(L, "rrtmgp_hip_reduce_fluxes_" + suf)(i(ncol), i(nlev), i(ngpt), i(0), None, up.ptr, dn.ptr,
                                                                 None, *[o.ptr for o in all_], *[None] * 5, None))
    for a, b in zip(one, all_):
        assert np.any(_host(a) != 0) and np.array_equal(_host(a), _host(b))
