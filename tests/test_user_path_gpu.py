"""The user-callable path's kernels at the sizes where they switch or can go
wrong: chunk and table edges, remainders, unaligned buffers."""
import ctypes

import numpy as np
import pytest
import torch

from torchquad_amd import _lib, _ops
from torchquad_amd.gl_nodes import gauss_legendre

pytestmark = pytest.mark.gpu


def _unaligned(count, dtype, dev):
    """A contiguous buffer of `count` elements one element past a 16-byte boundary."""
    return torch.full((count + 8,), float("nan"), dtype=dtype, device=dev)[1 : count + 1]


def _box(d, dtype, dev, seed=0):
    rng = np.random.default_rng(seed)
    b = np.stack([rng.uniform(-1, 0, d), rng.uniform(0.5, 2, d)], axis=1)
    return torch.tensor(b, dtype=dtype, device=dev)


# (dim, n): one point to a chunk's edge (64 and 256 points), odd totals, more
# axes than four points per lane take, axes too long for the node table
POINTS = [(1, 2), (1, 64), (1, 255), (1, 256), (1, 257), (1, 20011), (2, 16), (2, 17), (3, 7), (5, 5), (7, 3), (8, 3),
          (9, 2), (12, 2), (2, 2500)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["trapezoid", "gauss_legendre"])
@pytest.mark.parametrize("d,n", POINTS)
def test_grid_points_staged(d, n, rule, dtype, dev):
    dom = _box(d, dtype, dev, d + n)
    gl = gauss_legendre(n, device=dev) if rule == "gauss_legendre" else None
    pts = _ops.grid_points(_ops.RULES[rule], d, n, dom, gl)
    # the coordinate-by-coordinate kernel, which an unaligned output takes
    other = _unaligned(n**d * d, dtype, dev)
    g = _ops.grid_desc(_ops.RULES[rule], d, n, dtype, gl)
    _lib.call("tq_grid_points", ctypes.byref(g), _lib.ptr(dom), _lib.ptr(other), _lib.stream_ptr(dev))
    assert torch.equal(pts, other.view(n**d, d))
    # and the definition: x = lo + j h (or the mapped root), ij order
    b = dom.double()
    axes = []
    for k in range(d):
        lo, hi = b[k, 0], b[k, 1]
        if gl is not None:
            axes.append(0.5 * (hi - lo) * gl[0] + 0.5 * (hi + lo))
        else:
            axes.append(lo + torch.arange(n, dtype=torch.float64, device=dev) * ((hi - lo) / (n - 1)))
    ref = torch.stack([m.ravel() for m in torch.meshgrid(*axes, indexing="ij")], dim=1)
    # one rounding to the data type of values below 2, and a few of the FP64 reference
    tol = 2.0**-24 * 2 if dtype == torch.float32 else 2.0**-50
    assert float((pts.double() - ref).abs().max()) <= tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("d,N", [(1, 1), (1, 63), (2, 64), (3, 257), (4, 1024), (5, 999), (7, 130), (8, 4097),
                                 (9, 65), (16, 300)])
def test_mc_points_staged(d, N, dtype, dev):
    dom = _box(d, dtype, dev, N)
    pts = _ops.mc_points(d, N, dom, 1234567890123, 77)
    other = _unaligned(N * d, dtype, dev)
    m = _ops.mc_desc(d, N, dtype, 1234567890123, 77)
    _lib.call("tq_mc_points", ctypes.byref(m), _lib.ptr(dom), _lib.ptr(other), _lib.stream_ptr(dev))
    assert torch.equal(pts, other.view(N, d))
    lo, hi = dom[:, 0], dom[:, 1]
    assert bool(((pts >= lo) & (pts <= hi)).all())
