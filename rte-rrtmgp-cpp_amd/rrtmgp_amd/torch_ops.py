"""torch.autograd bindings of the column-radiation path.

No reference counterpart: the reference's Python binding (python/radiation.pyx) is forward only.
Forward passes run the library's HIP kernels (fused gas optics, cloud optics, solvers); backward
passes run its adjoint drivers (rrtmgp_api_adjoint_lw / _sw) and the heating-rate adjoint kernel.
torch only holds the tensors: they are copied device to device into the library's Fortran-order
arrays and back, the tensors of a call in one launch.

Shapes (tensors on the HIP device, any strides): profiles (ncol, nlay) or (ncol, nlev); t_sfc,
mu0 and tsi_scaling (ncol); surface emissivity and albedo (nbnd, ncol).  Gases other than h2o and
o3 come as a dict of constant vmr (scalars or (ncol, nlay) arrays) and receive no gradient;
clouds (lwp, iwp, rel, rei) are held fixed.
"""
from __future__ import annotations

import ctypes as C
from types import SimpleNamespace

import numpy as np
import torch

from . import _lib, api
from .device import DeviceArray, synchronize


def _np_dtype(precision):
    return np.float64 if precision == 8 else np.float32


def _torch_dtype(precision):
    return torch.float64 if precision == 8 else torch.float32


class _CopyItem(C.Structure):
    _fields_ = [("src", C.c_void_p), ("dst", C.c_void_p)] + [(n, C.c_int64) for n in ("n0", "n1", "s0", "s1")] + \
               [("src_size", C.c_int32), ("dst_size", C.c_int32)]


def _copy_all(items):
    """Runs the copies and returns when they are done."""
    c = (_CopyItem * len(items))(*items)
    _lib.check_hip(_lib.hip().rrtmgp_hip_copy_arrays(C.c_int(len(items)), c, None))
    synchronize()


def to_device_arrays(tensors, precision: int) -> list:
    """Copies device tensors (any strides) into new DeviceArrays of the same shapes (Fortran order)."""
    here = torch.device("cuda", torch.cuda.current_device())
    keep, out, items = [], [], []
    for t in tensors:
        x = t.detach().resolve_neg()
        if not x.is_cuda:
            raise ValueError(f"expected a device tensor, got one on {x.device}")
        if x.device != here or x.dtype not in (torch.float32, torch.float64) or x.dim() > 2:
            x = x.to(device=here, dtype=_torch_dtype(precision))
            x = x.permute(tuple(reversed(range(x.dim())))).contiguous().reshape(-1)     # Fortran order
        d = DeviceArray(tuple(t.shape), _np_dtype(precision), zero=False)
        n = tuple(x.shape) + (1, 1)
        s = x.stride() + (1, 1)
        items.append(_CopyItem(x.data_ptr(), d.ptr.value, n[0], n[1], s[0], s[1], x.element_size(), d.dtype.itemsize))
        keep.append(x)
        out.append(d)
    for device in {x.device for x in keep} | {t.device for t in tensors}:
        torch.cuda.synchronize(device)
    _copy_all(items)
    return out


def to_tensors(arrays, device) -> list:
    """Tensors of the DeviceArrays' shapes on `device` holding copies of them."""
    here = torch.device("cuda", torch.cuda.current_device())
    out = [torch.empty(tuple(reversed(d.shape)), dtype=torch.float64 if d.dtype == np.float64 else torch.float32,
                       device=here) for d in arrays]
    synchronize()
    _copy_all([_CopyItem(d.ptr.value, x.data_ptr(), d.size, 1, 1, 1, d.dtype.itemsize, d.dtype.itemsize)
               for d, x in zip(arrays, out)])
    return [x.to(device).permute(tuple(reversed(range(x.dim())))) for x in out]


def to_device_array(t: torch.Tensor, precision: int) -> DeviceArray:
    """Copy a device tensor into a new DeviceArray of the same shape (Fortran order)."""
    return to_device_arrays([t], precision)[0]


def to_tensor(d: DeviceArray, device) -> torch.Tensor:
    """A tensor of d's shape on `device` holding a copy of d."""
    return to_tensors([d], device)[0]


def _atmosphere(precision, ncol, nlay, arrays: dict, vmr: dict, clouds):
    """A DeviceAtmosphere-like namespace over device copies of the inputs."""
    a = SimpleNamespace(ncol=ncol, nlay=nlay, precision=precision)
    cloud_names = ("lwp", "iwp", "rel", "rei")
    on_device = dict(arrays)
    on_device.update({"vmr " + k: v for k, v in vmr.items() if isinstance(v, torch.Tensor)})
    if clouds is not None:
        on_device.update({k: clouds[k] for k in cloud_names})
    got = dict(zip(on_device, to_device_arrays(list(on_device.values()), precision)))
    for k in arrays:
        setattr(a, k, got[k])
    dev_vmr = {k: got["vmr " + k] if isinstance(v, torch.Tensor) else np.atleast_2d(np.asarray(v, _np_dtype(precision)))
               for k, v in vmr.items()}
    a.gas_concs = api.GasConcs(dev_vmr, precision)
    a._vmr = dev_vmr                                          # keeps the device copies alive
    a.cloudy = clouds is not None
    for k in cloud_names:
        setattr(a, k, got[k] if clouds is not None else None)
    return a


def _refuse_surrogate(solver):
    """The backward runs the adjoint of the plain gas optics; a forward through an MLP surrogate
    would pair fluxes of one function with gradients of another."""
    if getattr(solver.kd, "_surrogate", None) is not None:
        raise ValueError("autograd through a k-distribution with an MLP surrogate set is not supported: the "
                         "adjoint differentiates the plain gas optics; clear the surrogate first")


class _Longwave(torch.autograd.Function):
    @staticmethod
    def forward(ctx, solver, other_vmr, clouds, t_lay, t_lev, t_sfc, p_lay, p_lev, h2o, o3, emis_sfc):
        _refuse_surrogate(solver)
        ncol, nlay = t_lay.shape
        vmr = dict(other_vmr)
        vmr["h2o"], vmr["o3"] = h2o, o3
        da = _atmosphere(solver.precision, ncol, nlay,
                         {"t_lay": t_lay, "t_lev": t_lev, "t_sfc": t_sfc, "p_lay": p_lay, "p_lev": p_lev,
                          "emis_sfc": emis_sfc}, vmr, clouds)
        o = solver.solve(da)
        ctx.solver, ctx.da, ctx.dev = solver, da, t_lay.device
        ctx.save_for_backward(p_lay)
        return tuple(to_tensors([o["flux_up"], o["flux_dn"]], t_lay.device))

    @staticmethod
    def backward(ctx, g_up, g_dn):
        (p_lay,) = ctx.saved_tensors
        P = ctx.solver.precision
        g = ctx.solver.adjoint(ctx.da, *to_device_arrays([g_up, g_dn], P))
        t = dict(zip(g, to_tensors(list(g.values()), ctx.dev)))
        names = ctx.solver.kd.gas_names
        return (None, None, None, t["t_lay"], t["t_lev"], t["t_sfc"], t["lnp_lay"] / p_lay.to(t["lnp_lay"].dtype),
                t["p_lev"], t["vmr"][:, :, names.index("h2o")], t["vmr"][:, :, names.index("o3")], t["emis_sfc"])


class _Shortwave(torch.autograd.Function):
    @staticmethod
    def forward(ctx, solver, other_vmr, clouds, delta_cloud, mu0, tsi_scaling, t_lay, p_lay, p_lev, h2o, o3,
                sfc_alb):
        _refuse_surrogate(solver)
        ncol, nlay = t_lay.shape
        vmr = dict(other_vmr)
        vmr["h2o"], vmr["o3"] = h2o, o3
        P = solver.precision
        # t_lev is not read by the SW path; a copy of p_lev's shape keeps the interface uniform.
        da = _atmosphere(P, ncol, nlay, {"t_lay": t_lay, "t_lev": p_lev, "p_lay": p_lay, "p_lev": p_lev,
                                         "sfc_alb": sfc_alb, "mu0": mu0, "tsi": tsi_scaling}, vmr, clouds)
        tsi = da.tsi
        o = solver.solve(da, tsi, delta_cloud=delta_cloud)
        ctx.solver, ctx.da, ctx.tsi, ctx.delta, ctx.dev = solver, da, tsi, delta_cloud, t_lay.device
        ctx.save_for_backward(p_lay)
        return tuple(to_tensors([o[k] for k in ("flux_up", "flux_dn", "flux_dn_dir")], t_lay.device))

    @staticmethod
    def backward(ctx, g_up, g_dn, g_dir):
        (p_lay,) = ctx.saved_tensors
        P = ctx.solver.precision
        g = ctx.solver.adjoint(ctx.da, ctx.tsi, *to_device_arrays([g_up, g_dn, g_dir], P), delta_cloud=ctx.delta)
        t = dict(zip(g, to_tensors(list(g.values()), ctx.dev)))
        names = ctx.solver.kd.gas_names
        return (None, None, None, None, None, None, t["t_lay"], t["lnp_lay"] / p_lay.to(t["lnp_lay"].dtype),
                t["p_lev"], t["vmr"][:, :, names.index("h2o")], t["vmr"][:, :, names.index("o3")],
                t["sfc_alb_dir"] + t["sfc_alb_dif"])


class _HeatingRate(torch.autograd.Function):
    @staticmethod
    def forward(ctx, flux_up, flux_dn, p_lev, precision):
        ncol, nlev = flux_up.shape
        d = to_device_arrays([flux_up, flux_dn, p_lev], precision)
        hr = DeviceArray((ncol, nlev - 1), _np_dtype(precision))
        fn = getattr(_lib.hip(), "rrtmgp_hip_heating_rate_" + ("f64" if precision == 8 else "f32"))
        _lib.check_hip(fn(C.c_int64(ncol), C.c_int64(nlev - 1), d[0].ptr, d[1].ptr, d[2].ptr, hr.ptr, None))
        ctx.d, ctx.precision, ctx.dev = d, precision, flux_up.device
        return to_tensor(hr, flux_up.device)

    @staticmethod
    def backward(ctx, g_hr):
        P = ctx.precision
        up, dn, pl = ctx.d
        ncol, nlev = up.shape
        gu, gd, gp = (DeviceArray((ncol, nlev), _np_dtype(P)) for _ in range(3))
        gh = to_device_array(g_hr, P)
        fn = getattr(_lib.hip(), "rrtmgp_hip_heating_rate_adjoint_" + ("f64" if P == 8 else "f32"))
        _lib.check_hip(fn(C.c_int64(ncol), C.c_int64(nlev - 1), up.ptr, dn.ptr, pl.ptr, gh.ptr, gu.ptr, gd.ptr,
                          gp.ptr, None))
        return (*to_tensors([gu, gd, gp], ctx.dev), None)


def lw_fluxes(solver: api.SolverLW, t_lay, t_lev, t_sfc, p_lay, p_lev, h2o, o3, emis_sfc, other_vmr=None,
              clouds=None):
    """Broadband LW (flux_up, flux_dn) (ncol, nlev), differentiable in every tensor argument."""
    return _Longwave.apply(solver, other_vmr or {}, clouds, t_lay, t_lev, t_sfc, p_lay, p_lev, h2o, o3, emis_sfc)


def sw_fluxes(solver: api.SolverSW, t_lay, p_lay, p_lev, h2o, o3, sfc_alb, mu0, tsi_scaling, other_vmr=None,
              clouds=None, delta_cloud=True):
    """Broadband SW (flux_up, flux_dn, flux_dn_dir) (ncol, nlev); differentiable in t_lay, p_lay,
    p_lev, h2o, o3 and sfc_alb (used for the direct and the diffuse albedo)."""
    return _Shortwave.apply(solver, other_vmr or {}, clouds, delta_cloud, mu0, tsi_scaling, t_lay, p_lay, p_lev,
                            h2o, o3, sfc_alb)


def heating_rate(flux_up, flux_dn, p_lev, precision=8):
    """Heating rate (ncol, nlay) [K/day] of rrtmgp_hip_heating_rate_*, differentiable."""
    return _HeatingRate.apply(flux_up, flux_dn, p_lev, precision)
