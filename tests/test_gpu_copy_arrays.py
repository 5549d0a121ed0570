"""Strided copies between torch tensors and Fortran-order arrays, against torch: orders, steps, broadcast
strides and offsets, sizes around the 32 x 32 tiles, both element types in both directions, more arrays than
one launch takes, empty ones, and types that torch converts first.  Values are compared exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _variants(torch, shape):
    n, m = shape
    base = torch.randn(2 * n + 3, 2 * m + 3, device="cuda", dtype=torch.float64)
    yield base[:n, :m].contiguous()
    yield base[:n, :m].t().contiguous().t()
    yield base[1:n + 1, 2:m + 2]
    yield base[:2 * n:2, :2 * m:2]
    yield base[:2 * n:2, :m]
    yield base[:n, :1].expand(n, m)
    yield base[:1, :m].expand(n, m)
    yield base[:n, :m].float()
    yield base[:n, :m].t().float().t()
    yield base[:n, :m].half()
    yield (base[:n, :m] * 100).int()


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("shape", [(1, 1), (1, 40), (40, 1), (31, 33), (32, 32), (65, 7), (300, 129)])
def test_round_trip(precision, shape):
    torch = pytest.importorskip("torch")
    from rrtmgp_amd import torch_ops
    dt = torch.float64 if precision == 8 else torch.float32
    ts = list(_variants(torch, shape))
    ts += [ts[0][:, 0], ts[0][0], ts[3][:, 0], torch.tensor(3.25, device="cuda"), ts[0][:0], ts[0][:, :0],
           ts[0].reshape(shape + (1,)).expand(shape + (3,))]
    out = torch_ops.to_device_arrays(ts, precision)
    for t, d in zip(ts, out):
        want = t.to(dt).cpu().numpy()
        assert d.shape == want.shape and np.array_equal(d.to_host(), want)
    for t, x in zip(ts, torch_ops.to_tensors(out, ts[0].device)):
        assert x.dtype == dt and x.shape == t.shape and torch.equal(x, t.to(dt))


def test_host_tensor_is_refused():
    torch = pytest.importorskip("torch")
    from rrtmgp_amd import torch_ops
    with pytest.raises(ValueError):
        torch_ops.to_device_array(torch.zeros(3, 3), 8)


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("ncol,nlay", [(1, 1), (3, 2), (300, 17)])
def test_heating_rate_adjoint(precision, ncol, nlay):
    """The level-wise kernel against autograd of the formula; sums of a few terms, so a few eps of them."""
    torch = pytest.importorskip("torch")
    from rrtmgp_amd import torch_ops
    dt = torch.float64 if precision == 8 else torch.float32
    g = torch.Generator().manual_seed(ncol)
    up, dn = (100 + 300 * torch.rand(ncol, nlay + 1, generator=g, dtype=torch.float64) for _ in range(2))
    p = 1e5 - 1000 * (torch.arange(nlay + 1) + 0.4 * torch.rand(ncol, nlay + 1, generator=g, dtype=torch.float64))
    c = torch.randn(ncol, nlay, generator=g, dtype=torch.float64)
    x = [v.to(dt).cuda().requires_grad_() for v in (up, dn, p)]
    (torch_ops.heating_rate(*x, precision=precision) * c.to(dt).cuda()).sum().backward()
    y = [v.detach().double().cpu().requires_grad_() for v in x]
    net = y[1] - y[0]
    k = 9.80665 / 1004.64 * 86400.0
    (k * (net[:, :-1] - net[:, 1:]) / (y[2][:, 1:] - y[2][:, :-1]) * c.to(dt).double()).sum().backward()
    for a, b in zip(x, y):
        scale = b.grad.abs().max().item()
        assert (a.grad.cpu().double() - b.grad).abs().max().item() < 16 * torch.finfo(dt).eps * scale
