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
