"""Reverse mode of the gas optics for k-distributions of 19 and 32 gases (the most one may list): gradients
through the kernel ABI against central differences of the FP64 forward entry points, one band and a band range
a call; and the time of a call, which must hardly depend on gases that no absorber uses.

Half of the minor absorbers are moved to four further gases, of even and odd number and the last one among
them, some of them scaling each other.  Bar: as in the tests of the 5-gas k-distribution.
"""
import copy
import ctypes as C
import dataclasses
import time

import numpy as np
import pytest

from conftest import AVAILABLE
from test_gpu_adjoint import G, _host                           # noqa: F401  (G is a fixture)
from test_gpu_gas_optics_adjoint import DT, SIZES, Ctx, ragged

pytestmark = pytest.mark.gpu


def with_gases(kd, n):
    """The k-distribution with n gases, the further ones unused."""
    extra = [f"gas{i:02d}" for i in range(len(kd.gas_names) + 1, n + 1)]
    vr = np.asarray(kd.vmr_ref)
    ones = np.ones((vr.shape[0], len(extra), vr.shape[2]))
    return dataclasses.replace(kd, gas_names=list(kd.gas_names) + extra,
                               vmr_ref=np.asfortranarray(np.concatenate([vr, ones], axis=1))), extra


def use_gases(kd, extra):
    """Every second minor absorber moved to four of the further gases; returns them too."""
    kd = copy.deepcopy(kd)
    picks = [extra[0], extra[1], extra[-2], extra[-1]]
    kd.gas_minor = list(kd.gas_minor) + picks
    kd.identifier_minor = list(kd.identifier_minor) + picks
    for s in ("lower", "upper"):
        gases, scaling = list(getattr(kd, f"minor_gases_{s}")), list(getattr(kd, f"scaling_gas_{s}"))
        dens, compl = (np.array(getattr(kd, f"{f}_{s}")) for f in ("minor_scales_with_density", "scale_by_complement"))
        for i, m in enumerate(range(0, len(gases), 2)):
            gases[m], dens[m] = picks[i % 4], i % 3 != 2
            scaling[m], compl[m] = (picks[(i + 1) % 4], i % 4 == 0) if i % 2 == 0 and dens[m] else ("", 0)
        for f, v in (("minor_gases", gases), ("scaling_gas", scaling), ("minor_scales_with_density", dens),
                     ("scale_by_complement", compl)):
            setattr(kd, f"{f}_{s}", v)
    return kd, picks


class ManyGases(Ctx):
    """Ctx with the further gases, those in use among the differentiated inputs."""

    def __init__(self, G, syn, k, kd, lw, extra, used=()):
        super().__init__(G, syn, k, kd, lw, False)
        shape = (self.n, self.nlay)
        self.used = list(used)
        for name in extra:
            v = self.rng.uniform(1e-7, 1e-5, shape)
            (self.x if name in self.used else self.fixed)[name] = v

    def check(self, loss, grads):
        used, x = self.used, self.x
        names = [n for n in x if n not in used]
        self.x = {n: x[n] for n in names}
        full = lambda y: loss({**x, **y})                       # noqa: E731
        super().check(full, grads)
        self.x = x
        h = 1e-5
        for name in used:
            g = grads[0][:, :, self.k.gas_names.index(name) + 1] * self.cd
            assert np.abs(g).max() > 0, name
            v = self.rng.normal(size=g.shape) * 1e-2 * x[name]
            terms = [np.concatenate([t.ravel() for t in full({name: x[name] + e * v})]) for e in (h, -h)]
            fd = np.sum(terms[0] - terms[1]) / (2 * h)
            noise = 4 * np.finfo(DT).eps * np.linalg.norm(terms[0]) / h
            ad = np.sum(g * v)
            assert abs(ad - fd) <= 1e-7 * np.sum(np.abs(g * v)) + 3 * noise, (name, ad, fd, noise)


def _ctx(G, syn, kd, lw, n):
    k, extra = with_gases(kd, n)
    k, picks = use_gases(ragged(k), extra)
    return ManyGases(G, syn, k, G.KDist(k, AVAILABLE + extra, 8), lw, extra, picks)


@pytest.mark.parametrize("n", [19, 32])
@pytest.mark.parametrize("lw", [True, False])
def test_one_band(G, syn, kd_lw, kd_sw, lw, n):
    c = _ctx(G, syn, kd_lw if lw else kd_sw, lw, n)
    out, losses = c.outputs(), []
    for b in range(len(SIZES)):
        f = c.forward(c.x, b, 1, False)
        cot, dc = c.cotangents([v.shape for v in f[:5]], [max(np.abs(v).mean(), 1e-3) for v in f[:5]])
        a, keep = c.inputs(c.x)
        head = [C.c_int64(b), C.c_int64(c.n), C.c_int64(c.nlay)]
        if lw:
            c.call("gas_optics_lw_adjoint", *head, *a, *[v.ptr for v in dc], *[o.ptr for o in out])
        else:
            c.call("gas_optics_sw_adjoint", *head, *a, None, None, None, *[v.ptr for v in dc], *[o.ptr for o in out])
        losses.append((b, cot))
    c.check(lambda x: [q * v for b, cot in losses for q, v in zip(cot, c.forward(x, b, 1, False))],
            [_host(o) for o in out])


@pytest.mark.parametrize("n", [19, 32])
@pytest.mark.parametrize("lw", [True, False])
def test_band_range(G, syn, kd_lw, kd_sw, lw, n):
    c = _ctx(G, syn, kd_lw if lw else kd_sw, lw, n)
    nb = len(SIZES)
    out = c.outputs()
    f = c.forward(c.x, 0, nb, True)
    groups = [b for b in range(nb) for _ in range((SIZES[b] + 15) // 16)]
    a, keep = c.inputs(c.x)
    head = [C.c_int64(0), C.c_int64(nb), C.c_int64(c.n), C.c_int64(c.nlay)]
    if lw:
        gl = (c.n, c.nlay, len(groups))
        cot, dc = c.cotangents([f[0].shape, f[1].shape, gl, gl, gl, f[4].shape],
                               [f[0].mean(), f[1].mean(), f[2].mean(), f[2].mean(), f[2].mean(), f[4].mean()])
        c.call("gas_optics_lw_adjoint_bands", *head, *a, *[v.ptr for v in dc], *[o.ptr for o in out])
    else:
        cot, dc = c.cotangents([f[0].shape] * 2, [f[0].mean(), (f[0] * f[1]).mean()])
        c.call("gas_optics_sw_adjoint_bands", *head, *a, *[v.ptr for v in dc], *[o.ptr for o in out])

    def loss(x):
        f = c.forward(x, 0, nb, True)
        if lw:
            f = [f[0], f[1], f[2][:, :, groups], f[3][:, :-1][:, :, groups], f[3][:, 1:][:, :, groups], f[4]]
        else:
            f = [f[0] * (1.0 - f[1]), f[0] * f[1]]
        return [q * v for q, v in zip(cot, f)]

    c.check(loss, [_host(o) for o in out])


class Wide:
    """Atmospheres of enough columns to fill the GPU in place of Ctx's small one."""

    def __init__(self, syn):
        self.syn = syn

    def make_atmosphere(self, seed, ncol, nlay):
        return self.syn.make_atmosphere(seed, 8192, 64)


@pytest.mark.parametrize("bands", [1, 4])
@pytest.mark.parametrize("lw", [True, False])
def test_time_of_unused_gases(G, syn, kd_lw, kd_sw, lw, bands):
    """19 gases take at most 1.25 times as long as 5 (1.03 to 1.06 measured; with gradient rows per wavefront
    1.3 to 2.4): the shortest of five means of five calls each."""
    from rrtmgp_amd import device
    took = {}
    for n in (5, 19):
        k, extra = with_gases(kd_lw if lw else kd_sw, n)
        c = ManyGases(G, Wide(syn), k, G.KDist(k, AVAILABLE + extra, 8), lw, extra)
        ng = 16 * bands
        full, flat = (c.n, c.nlay, ng), (c.n, c.nlay, bands)
        if bands == 1:
            name, shapes, head = "adjoint", [full] * (4 if lw else 3), [C.c_int64(3)]
        else:
            name, shapes, head = "adjoint_bands", [full] * 2 + ([flat] * 3 if lw else []), [C.c_int64(2), C.c_int64(bands)]
        _, cot = c.cotangents(shapes + ([(c.n, ng)] if lw else []), [1.0] * 6)
        a, keep = c.inputs(c.x)
        out = c.outputs()
        args = head + [C.c_int64(c.n), C.c_int64(c.nlay)] + a + ([None] * 3 if bands == 1 and not lw else [])
        args += [v.ptr for v in cot] + [o.ptr for o in out]
        name = f"gas_optics_{'lw' if lw else 'sw'}_{name}"
        best = np.inf
        for _ in range(6):
            device.synchronize()
            t0 = time.perf_counter()
            for _ in range(5):
                c.call(name, *args)
            device.synchronize()
            best = min(best, time.perf_counter() - t0)
        took[n] = best
    assert took[19] <= 1.25 * took[5], took
