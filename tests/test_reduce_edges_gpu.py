"""Weighted sums of user values and their backward where the general form
degenerates: one node per axis, gradients at one end of an axis."""
import ctypes

import pytest
import torch

from torchquad_amd import _lib, _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("d,S", [(1, 1), (2, 1), (3, 1), (7, 1), (3, 5), (2, 70)])
def test_one_gauss_node_per_axis(d, S, dtype, dev):
    """The only point weighs w^d, forward and backward."""
    w = 1.5
    gl = (torch.tensor([0.25], dtype=torch.float64, device=dev), torch.tensor([w], dtype=torch.float64, device=dev))
    rule = _ops.RULES["gauss_legendre"]
    dom = torch.tensor([[-0.5, 1.0], [0.25, 2.0]] * 4, dtype=dtype, device=dev)[:d].contiguous()
    scale = float(torch.prod(0.5 * (dom[:, 1] - dom[:, 0]).double())) * w**d
    vals = torch.arange(1, S + 1, dtype=dtype, device=dev).reshape(1, S)
    # products of 2 d + 1 exact factors, one rounding to the data type
    eps = 2.0**-23 if dtype == torch.float32 else (2 * d + 2) * 2.0**-52
    out = _ops.grid_reduce(rule, d, 1, dom, vals, gl=gl)
    assert bool(((out.double() - scale * vals[0].double()).abs() <= eps * scale * vals[0].double()).all())
    g = torch.linspace(1.0, 2.0, S, dtype=dtype, device=dev)
    ref = scale * g.double()[None, :]
    gf, _ = _ops.grid_reduce_vjp(rule, d, 1, dom, g, out, 1, gl=gl)
    assert bool(((gf.double() - ref).abs() <= eps * ref).all())
    gf = _ops.grid_reduce_backward(rule, d, 1, dom, g, 1, gl=gl)
    assert bool(((gf.double() - ref).abs() <= eps * ref).all())
    # unaligned output: one value per store
    other = torch.full((S + 8,), float("nan"), dtype=dtype, device=dev)[1 : S + 1]
    desc = _ops.grid_desc(rule, d, 1, dtype, gl)
    _lib.call("tq_grid_reduce_backward", ctypes.byref(desc), _lib.ptr(dom), None, 0, _lib.ptr(g), S, _lib.ptr(other),
              _lib.stream_ptr(dev))
    assert bool(((other.double() - ref[0]).abs() <= eps * ref[0]).all())


@pytest.mark.parametrize("rule", ["trapezoid", "gauss_legendre"])
@pytest.mark.parametrize("d,n", [(1, 1001), (2, 31), (1, 3001)])
def test_points_backward_at_the_upper_end(d, n, rule, dev):
    """d/d lower bound takes g (1 - t) of every point: values 1e15 times as
    large at t = 1 do not blur it (Newton-Cotes: t is 1 there exactly)."""
    if rule == "gauss_legendre":
        t = torch.linspace(0.0, 1.0, n, dtype=torch.float64, device=dev)
        gl = (2.0 * t - 1.0, torch.ones_like(t))
    else:
        t, gl = torch.arange(n, dtype=torch.float64, device=dev) / (n - 1), None
    dom = torch.tensor([[-0.5, 1.0]] * d, dtype=torch.float64, device=dev)
    g = torch.ones([n] * d + [d], dtype=torch.float64, device=dev)
    for k in range(d):
        g.select(k, n - 1)[..., k] = 1e15
    got = _ops.grid_points_backward(_ops.RULES[rule], d, n, dom, g.reshape(-1, d).contiguous(), gl)
    for k in range(d):
        rows = g[..., k].sum(dim=[q for q in range(d) if q != k]) if d > 1 else g[..., 0]
        ref = float(torch.sum(rows * (1.0 - t)))
        # a sum of n^d terms of one sign, t to half a unit in the last place
        assert abs(float(got[k, 0]) - ref) <= (n**d + 4) * 2.0**-53 * ref
