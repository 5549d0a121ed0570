"""Reverse mode of the gas optics through the kernel ABI, against central differences of the FP64
forward entry points: one band per call with the cotangents of all outputs
(rrtmgp_hip_gas_optics_{lw,sw}_adjoint_*), and a band range with factored sources or gas optical depths
(rrtmgp_hip_gas_optics_{lw,sw}_adjoint_bands_*); and the drivers' gradients on the same k-distribution.

The k-distribution has bands of 16, 5, 20, 1, 33 and 16 g-points: full and partial 16-g-point chunks,
quads that end inside a band, and bands of two and three chunks.  65 columns fill one tile and start
another.

Bar: 1e-7 of sum |gradient x direction| (the step h = 1e-5 leaves h^2 = 1e-10 of truncation) plus what the
outputs' rounding puts into the quotient: a loss of terms c_i f_i, each f_i off by up to ~4 eps in either
evaluation, moves by 4 eps sqrt(sum (c_i f_i)^2) / h (a few times that at three standard deviations).
"""
import copy
import ctypes as C

import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_adjoint import G, _directions, _dot, _host, _perturbed   # noqa: F401  (G is a fixture)

pytestmark = pytest.mark.gpu

SIZES = [16, 5, 20, 1, 33, 16]
DT = np.float64
INT_FIELDS = ("ngas", "nflav", "neta", "npres", "ntemp", "ngpt", "nbnd", "nplanck", "idx_h2o")
REAL_FIELDS = ("press_ref_log_delta", "temp_ref_min", "temp_ref_delta", "press_ref_trop_log", "totplnk_delta")
PTR_FIELDS = ("flavor", "gpoint_flavor", "band_lims_gpt", "press_ref_log", "temp_ref", "vmr_ref", "kmajor",
              "kminor_lower", "kminor_upper", "minor_limits_gpt_lower", "minor_limits_gpt_upper",
              "minor_scales_with_density_lower", "minor_scales_with_density_upper", "scale_by_complement_lower",
              "scale_by_complement_upper", "idx_minor_lower", "idx_minor_upper", "idx_minor_scaling_lower",
              "idx_minor_scaling_upper", "kminor_start_lower", "kminor_start_upper", "totplnk", "planck_frac", "krayl")


class KdistDev(C.Structure):
    _fields_ = ([(n, C.c_int64) for n in INT_FIELDS] + [(n, C.c_double) for n in REAL_FIELDS]
                + [("nminor_lower", C.c_int64), ("nminor_upper", C.c_int64)] + [(n, C.c_void_p) for n in PTR_FIELDS]
                + [("ncontrib_lower", C.c_int64), ("ncontrib_upper", C.c_int64)]
                + [(n, C.c_void_p) for n in ("go_bands", "kmajor_p", "planck_frac_p", "kminor_p", "krayl_p")]
                + [("max_band_gpts", C.c_int64)])


class GasVmr(C.Structure):
    _fields_ = [("ngas", C.c_int64), ("vmr", C.c_void_p * 32), ("dim1", C.c_int64 * 32), ("dim2", C.c_int64 * 32)]


def ragged(kd):
    """The first bands of a synthetic k-distribution (16 g-points each) cut and repeated to SIZES."""
    nb = len(SIZES)
    pick = np.concatenate([16 * b + np.arange(n) % 16 for b, n in enumerate(SIZES)])
    end = np.cumsum(SIZES)
    k = copy.deepcopy(kd)
    k.band2gpt = np.asfortranarray(np.stack([end - np.array(SIZES) + 1, end]).astype(np.int32))
    k.key_species = np.asfortranarray(kd.key_species[:, :, :nb])
    k.band_lims_wavenum = np.asfortranarray(kd.band_lims_wavenum[:, :nb])
    k.kmajor = np.asfortranarray(kd.kmajor[pick])
    for s in ("lower", "upper"):
        lim, start = getattr(kd, f"minor_limits_gpt_{s}"), getattr(kd, f"kminor_start_{s}")
        keep = [m for m in range(lim.shape[1]) if (lim[0, m] - 1) // 16 < nb]
        rows, limits, starts = [], [], []
        for m in keep:
            b = (lim[0, m] - 1) // 16
            starts.append(sum(len(r) for r in rows) + 1)
            rows.append(start[m] - 1 + np.arange(SIZES[b]) % 16)
            limits.append(k.band2gpt[:, b])
        setattr(k, f"kminor_{s}", np.asfortranarray(getattr(kd, f"kminor_{s}")[np.concatenate(rows)]))
        setattr(k, f"minor_limits_gpt_{s}", np.asfortranarray(np.array(limits, dtype=np.int32).T))
        setattr(k, f"kminor_start_{s}", np.array(starts, dtype=np.int32))
        for f in ("minor_gases", "scaling_gas"):
            setattr(k, f"{f}_{s}", [getattr(kd, f"{f}_{s}")[m] for m in keep])
        for f in ("minor_scales_with_density", "scale_by_complement"):
            setattr(k, f"{f}_{s}", getattr(kd, f"{f}_{s}")[keep])
    if kd.is_lw:
        k.totplnk = np.asfortranarray(kd.totplnk[:, :nb])
        k.planck_frac = np.asfortranarray(kd.planck_frac[pick])
    else:
        for f in ("solar_src_quiet", "solar_src_facular", "solar_src_sunspot", "rayl_lower", "rayl_upper"):
            setattr(k, f, np.asfortranarray(getattr(kd, f)[pick]))
    return k


class Tables:
    """The device form of a k-distribution (every gas available), as the class layer uploads it."""

    def __init__(self, G, k, kd):
        from rrtmgp_amd import _lib
        self.L, self.keep, d = _lib.hip(), [], KdistDev()
        dev = lambda a, t=DT: self.keep.append(G.DeviceArray.from_host(np.asfortranarray(a), t)) or self.keep[-1].ptr.value  # noqa: E731
        nb, nt = k.nbnd, k.temp_ref.size
        flavor = kd.get_int("flavor")
        d.ngas, d.nflav, d.neta, d.npres, d.ntemp = len(k.gas_names), flavor.size // 2, k.kmajor.shape[1], k.press_ref.size, nt
        d.ngpt, d.nbnd, d.nplanck, d.idx_h2o = k.ngpt, nb, (k.totplnk.shape[0] if k.is_lw else 0), 1
        lp = np.log(k.press_ref)
        d.press_ref_log_delta, d.press_ref_trop_log = (lp[-1] - lp[0]) / (lp.size - 1), np.log(k.press_ref_trop)
        d.temp_ref_min, d.temp_ref_delta = k.temp_ref[0], (k.temp_ref[-1] - k.temp_ref[0]) / (nt - 1)
        d.totplnk_delta = (k.temp_ref[-1] - k.temp_ref[0]) / (d.nplanck - 1) if k.is_lw else 0.0
        d.flavor, d.gpoint_flavor = dev(flavor, np.int32), dev(kd.get_int("gpoint_flavor"), np.int32)
        d.band_lims_gpt = dev(k.band2gpt, np.int32)
        d.press_ref_log, d.temp_ref, d.vmr_ref = dev(lp), dev(k.temp_ref), dev(k.vmr_ref)
        d.kmajor = dev(k.kmajor.transpose(3, 1, 2, 0))
        for s in ("lower", "upper"):
            km = getattr(k, f"kminor_{s}")
            setattr(d, f"nminor_{s}", len(getattr(k, f"minor_gases_{s}")))
            setattr(d, f"ncontrib_{s}", km.shape[0])
            setattr(d, f"kminor_{s}", dev(km.transpose(2, 1, 0)))
            setattr(d, f"minor_limits_gpt_{s}", dev(getattr(k, f"minor_limits_gpt_{s}"), np.int32))
            for f in ("minor_scales_with_density", "scale_by_complement"):
                setattr(d, f"{f}_{s}", dev(getattr(k, f"{f}_{s}"), np.int8))
            for f in ("idx_minor", "idx_minor_scaling", "kminor_start"):
                setattr(d, f"{f}_{s}", dev(kd.get_int(f"{f}_{s}"), np.int32))
        if k.is_lw:
            d.totplnk, d.planck_frac = dev(k.totplnk), dev(k.planck_frac.transpose(3, 1, 2, 0))
        else:
            d.krayl = dev(np.stack([k.rayl_lower.transpose(2, 1, 0), k.rayl_upper.transpose(2, 1, 0)], axis=3))
        pack = C.c_void_p()
        _lib.check_hip(self.L.rrtmgp_hip_kdist_pack_f64(C.byref(d), C.byref(pack)))
        self.d, self.pack = d, pack

    def __del__(self):
        self.L.rrtmgp_hip_kdist_pack_free(self.pack)


class Ctx:
    """Calls of the ABI on one atmosphere; x holds the differentiated inputs."""

    def __init__(self, G, syn, k, kd, lw, cloud):
        self.G, self.t, self.lw, self.k = G, Tables(G, k, kd), lw, k
        atm = syn.make_atmosphere(71, 65, 3)
        self.n, self.nlay = atm.p_lay.shape
        rng = np.random.default_rng(8)
        self.x = {"t": atm.t_lay, "lnp": np.log(atm.p_lay), "h2o": atm.vmr["h2o"], "o3": atm.vmr["o3"]}
        if lw:
            self.x.update(tlev=atm.t_lev, tsfc=atm.t_sfc)
        self.fixed = {g: np.full((self.n, self.nlay), atm.vmr[g][0, 0]) for g in AVAILABLE if g not in ("h2o", "o3")}
        self.cd = 2.1e25 * rng.uniform(0.5, 1.5, (self.n, self.nlay)) / self.nlay
        self.cloud = [rng.uniform(0.1, 2.0, (self.n, self.nlay, k.nbnd)) * s for s in (1.0, 0.45, 0.4)] if cloud else None
        self.rng = rng

    def dev(self, a):
        return self.G.DeviceArray.from_host(np.asfortranarray(a), DT)

    def inputs(self, x):
        """Device arrays (kept alive by the caller) and the leading call arguments after (kd, bands, ncol, nlay)."""
        g = GasVmr()
        keep = []
        g.ngas = len(self.k.gas_names)
        for i, name in enumerate(self.k.gas_names):
            keep.append(self.dev(x[name] if name in x else self.fixed[name]))
            g.vmr[i], g.dim1[i], g.dim2[i] = keep[-1].ptr.value, self.n, self.nlay
        p, t, cd = self.dev(np.exp(x["lnp"])), self.dev(x["t"]), self.dev(self.cd)
        keep += [g, p, t, cd]
        a = [p.ptr, t.ptr]
        if self.lw:
            tl, ts = self.dev(x["tlev"]), self.dev(x["tsfc"])
            keep += [tl, ts]
            a += [tl.ptr, ts.ptr]
        a += [cd.ptr, C.byref(g)]
        if self.lw:
            a.append(C.c_int(1))
        return a, keep

    def call(self, name, *args):
        from rrtmgp_amd import _lib
        _lib.check_hip(getattr(self.t.L, f"rrtmgp_hip_{name}_f64")(C.byref(self.t.d), *args, None))

    def new(self, *shape):
        return self.G.DeviceArray(shape, DT)

    def forward(self, x, b0, nb, factored):
        ng = sum(SIZES[b0:b0 + nb])
        a, keep = self.inputs(x)
        i = C.c_int64
        head = [i(b0), i(nb), i(self.n), i(self.nlay)]
        shape = (self.n, self.nlay, ng)
        if self.lw and factored:
            o = [self.new(*shape), self.new(*shape), self.new(self.n, self.nlay, nb), self.new(self.n, self.nlay + 1, nb),
                 self.new(self.n, ng), self.new(self.n, ng)]
            self.call("gas_optics_lw_bands_factored", *head, *a, None, *[v.ptr for v in o])
        elif self.lw:
            o = [self.new(*shape) for _ in range(4)] + [self.new(self.n, ng), self.new(self.n, ng)]
            self.call("gas_optics_lw_bands", *head, *a, None, *[v.ptr for v in o])
        else:
            cl = [self.dev(c) for c in self.cloud] if self.cloud else []
            o = [self.new(*shape) for _ in range(3)]
            self.call("gas_optics_sw_bands", *head, *a, *([c.ptr for c in cl] or [None] * 3), *[v.ptr for v in o])
        return [_host(v) for v in o]

    def check(self, loss, grads):
        """grads: d_col (ncol, nlay, ngas + 2), d_t, d_lnp (, d_lo, d_hi, d_tsfc) against differences of the sum
        of the terms that loss(x) returns."""
        d_col, d_t, d_lnp = grads[:3]
        ih, io = (self.k.gas_names.index(g) + 1 for g in ("h2o", "o3"))
        g = {"t": d_t, "lnp": d_lnp, "h2o": d_col[:, :, ih] * self.cd, "o3": d_col[:, :, io] * self.cd}
        if self.lw:
            lev = np.zeros((self.n, self.nlay + 1))
            lev[:, :-1] += grads[3]
            lev[:, 1:] += grads[4]
            g.update(tlev=lev, tsfc=grads[5])
        h = 1e-5
        size = {"t": 1.0, "lnp": 1e-2, "tlev": 1.0, "tsfc": 1.0}
        for name, x in self.x.items():
            v = self.rng.normal(size=x.shape) * size.get(name, 1e-2 * x)
            terms = [np.concatenate([t.ravel() for t in loss({**self.x, name: x + e * v})]) for e in (h, -h)]
            fd = np.sum(terms[0] - terms[1]) / (2 * h)
            noise = 4 * np.finfo(DT).eps * np.linalg.norm(terms[0]) / h
            ad = np.sum(g[name] * v)
            assert abs(ad - fd) <= 1e-7 * np.sum(np.abs(g[name] * v)) + 3 * noise, (name, ad, fd, noise)

    def outputs(self):
        ng = len(self.k.gas_names)
        o = [self.new(self.n, self.nlay, ng + 2), self.new(self.n, self.nlay), self.new(self.n, self.nlay)]
        return o + ([self.new(self.n, self.nlay), self.new(self.n, self.nlay), self.new(self.n)] if self.lw else [])

    def cotangents(self, shapes, scales):
        c = [self.rng.normal(size=s) / v for s, v in zip(shapes, scales)]
        return c, [self.dev(a) for a in c]


@pytest.mark.parametrize("lw,cloud", [(True, False), (False, False), (False, True)])
def test_one_band_adjoint(G, syn, kd_lw, kd_sw, lw, cloud):
    k = ragged(kd_lw if lw else kd_sw)
    c = Ctx(G, syn, k, G.KDist(k, AVAILABLE, 8), lw, cloud)
    out, losses = c.outputs(), []
    for b in range(k.nbnd):
        f = c.forward(c.x, b, 1, False)
        cot, dc = c.cotangents([v.shape for v in f[:5]], [max(np.abs(v).mean(), 1e-3) for v in f[:5]])
        a, keep = c.inputs(c.x)
        head = [C.c_int64(b), C.c_int64(c.n), C.c_int64(c.nlay)]
        if lw:
            c.call("gas_optics_lw_adjoint", *head, *a, *[v.ptr for v in dc], *[o.ptr for o in out])
        else:
            cl = [c.dev(v) for v in c.cloud] if cloud else []
            c.call("gas_optics_sw_adjoint", *head, *a, *([v.ptr for v in cl] or [None] * 3), *[v.ptr for v in dc],
                   *[o.ptr for o in out])
        losses.append((b, cot))
    c.check(lambda x: [q * v for b, cot in losses for q, v in zip(cot, c.forward(x, b, 1, False))],
            [_host(o) for o in out])


@pytest.mark.parametrize("lw", [True, False])
def test_band_range_adjoint(G, syn, kd_lw, kd_sw, lw):
    k = ragged(kd_lw if lw else kd_sw)
    c = Ctx(G, syn, k, G.KDist(k, AVAILABLE, 8), lw, False)
    out, losses = c.outputs(), []
    for b0, nb in ((0, 4), (4, 2)):
        f = c.forward(c.x, b0, nb, True)
        a, keep = c.inputs(c.x)
        head = [C.c_int64(b0), C.c_int64(nb), C.c_int64(c.n), C.c_int64(c.nlay)]
        groups = [b for b in range(nb) for _ in range((SIZES[b0 + b] + 15) // 16)]
        if lw:
            gl = (c.n, c.nlay, len(groups))
            cot, dc = c.cotangents([f[0].shape, f[1].shape, gl, gl, gl, f[4].shape],
                                   [f[0].mean(), f[1].mean(), f[2].mean(), f[2].mean(), f[2].mean(), f[4].mean()])
            c.call("gas_optics_lw_adjoint_bands", *head, *a, *[v.ptr for v in dc], *[o.ptr for o in out])
        else:
            cot, dc = c.cotangents([f[0].shape] * 2, [f[0].mean(), (f[0] * f[1]).mean()])
            c.call("gas_optics_sw_adjoint_bands", *head, *a, *[v.ptr for v in dc], *[o.ptr for o in out])
        losses.append((b0, nb, groups, cot))

    def loss(x):
        s = []
        for b0, nb, groups, cot in losses:
            f = c.forward(x, b0, nb, True)
            if lw:
                f = [f[0], f[1], f[2][:, :, groups], f[3][:, :-1][:, :, groups], f[3][:, 1:][:, :, groups], f[4]]
            else:
                f = [f[0] * (1.0 - f[1]), f[0] * f[1]]
            s += [q * v for q, v in zip(cot, f)]
        return s

    c.check(loss, [_host(o) for o in out])


@pytest.mark.parametrize("lw", [True, False])
def test_drivers_on_ragged_bands(G, O, syn, kd_lw, kd_sw, lut_lw, lut_sw, lw):
    """End to end against the oracle (1e-5, as the other end-to-end tests)."""
    k = ragged(kd_lw if lw else kd_sw)
    lut = copy.deepcopy(lut_lw if lw else lut_sw)
    nb = len(SIZES)
    for f in ("band_lims_wvn", "lut_extliq", "lut_ssaliq", "lut_asyliq", "lut_extice", "lut_ssaice", "lut_asyice"):
        setattr(lut, f, np.asfortranarray(getattr(lut, f)[:, :nb]))
    atm = syn.make_atmosphere(53, 5, 30, cloudy=True, nbnd_lw=nb, nbnd_sw=nb)
    kd, okd = G.KDist(k, AVAILABLE, 8), O.Kdist(k, AVAILABLE)
    rng = np.random.default_rng(13)
    a = [rng.normal(size=(atm.ncol, atm.nlay + 1)) for _ in range(2 if lw else 3)]
    da = G.DeviceAtmosphere(atm, 8)
    if lw:
        grad = G.SolverLW(kd, G.Cloud(lut, 8)).adjoint(da, *a)
    else:
        tsi = np.full(atm.ncol, atm.tsi / kd.scalar("tsi"))
        grad = G.SolverSW(kd, G.Cloud(lut, 8)).adjoint(da, tsi, *a)
    grad = {n: _host(d) for n, d in grad.items()}

    def loss(at):
        o = O.solve_lw(okd, at, O.Cloud(lut)) if lw else O.solve_sw(okd, at, O.Cloud(lut), tsi_scaling=tsi)
        return float(sum(np.sum(q * o[n]) for q, n in zip(a, ("flux_up", "flux_dn", "flux_dn_dir"))))

    v = _directions(rng, atm, lw)
    h = 1e-4
    fd = (loss(_perturbed(atm, v, h)) - loss(_perturbed(atm, v, -h))) / (2 * h)
    ad = _dot(G, grad, v, kd.gas_names, lw)
    assert abs(ad - fd) <= 1e-5 * abs(fd), (ad, fd)


@pytest.mark.parametrize("thin", [False, True])
def test_shortwave_chains_agree_in_cloud(G, syn, kd_sw, thin):
    """Reverse mode of solver and gas optics through the gases' optical depths against the chain through tau, ssa
    and g, with clouds in every layer.  Where a layer's gases are thinner than the combine rule's cut-off
    (2 eps), Rayleigh scattering does not reach the fluxes, however thick the cloud.  Bar: both chains evaluate
    the same derivatives in FP64, 1e-9 of a layer's largest."""
    k = ragged(kd_sw)
    c = Ctx(G, syn, k, G.KDist(k, AVAILABLE, 8), False, True)
    if thin:
        c.cd[::3, 1] = 1e3                       # molecules per cm2: optical depths of 1e-20 and less
        c.cd[1::3, 2] = 1e9
    nb, ng = len(SIZES), sum(SIZES)
    full, lev, bnd = (c.n, c.nlay, ng), (c.n, c.nlay + 1), (c.n, ng)
    a, keep = c.inputs(c.x)
    i = C.c_int64
    size, cl = [i(c.n), i(c.nlay)], [c.dev(v) for v in c.cloud]
    opt = [c.new(*full) for _ in range(3)]
    c.call("gas_optics_sw_bands", i(0), i(nb), *size, *a, *[v.ptr for v in cl], *[v.ptr for v in opt])
    rng = np.random.default_rng(4)
    mu0, alb, inc = c.dev(rng.uniform(0.2, 1, c.n)), c.dev(rng.uniform(0.1, 0.5, bnd)), c.dev(rng.uniform(1, 2, bnd))
    cot = [c.dev(rng.normal(size=lev)) for _ in range(3)]
    args = size + [i(ng), C.c_int(0)] + [v.ptr for v in (*opt, mu0, alb, alb, inc)] + [None] + [v.ptr for v in cot]
    alb_out = [c.new(*bnd) for _ in range(2)]

    def solver(name, out):
        from rrtmgp_amd import _lib
        _lib.check_hip(getattr(c.t.L, f"rrtmgp_hip_{name}_f64")(*args, *[v.ptr for v in out + alb_out], None))

    d3, d2 = [c.new(*full) for _ in range(3)], [c.new(*full) for _ in range(2)]
    solver("sw_solver_2stream_adjoint", d3)
    solver("sw_adjoint_gases", d2)
    one, two = c.outputs(), c.outputs()
    g0 = 0
    for b, n in enumerate(SIZES):
        part = [c.dev(_host(v)[:, :, g0:g0 + n]) for v in d3]
        c.call("gas_optics_sw_adjoint", i(b), *size, *a, *[v.ptr for v in cl], *[v.ptr for v in part], *[o.ptr for o in one])
        g0 += n
    c.call("gas_optics_sw_adjoint_bands", i(0), i(nb), *size, *a, *[v.ptr for v in d2], *[o.ptr for o in two])
    for name, x, y in zip(("d_col", "d_t", "d_lnp"), one, two):
        x, y = (_host(v).reshape(c.n, c.nlay, -1) for v in (x, y))
        scale = np.abs(x).max(axis=0)            # per layer and gas: gradients of a thin layer are of another size
        assert (np.abs(x - y) <= 1e-9 * scale).all(), (name, (np.abs(x - y) / np.maximum(scale, 1e-300)).max())
