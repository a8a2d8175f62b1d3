"""The user path's kernels on both sides of the sizes where their launches
change: points per lane and the node table of the writers, the direct and the
tabulated weights and the waves' spans of the backward, the final sum's block."""
import ctypes

import numpy as np
import pytest
import torch

from torchquad_amd import _lib, _ops
from torchquad_amd.gl_nodes import gauss_legendre

pytestmark = pytest.mark.gpu

M = 1 << 19  # values from which the backward takes tables; FP32 points from which a grid's lane takes four


def _unaligned(count, dtype, dev):
    """A contiguous buffer of `count` elements one element past a 16-byte boundary."""
    return torch.full((count + 8,), float("nan"), dtype=dtype, device=dev)[1 : count + 1]


def _box(d, dtype, dev):
    return torch.tensor([[-0.3, 1.1], [0.2, 0.9]] * 4, dtype=dtype, device=dev)[:d].contiguous()


# just below and above 2^18 (FP64) and 2^19 (FP32) points, with and without the node table, last chunks of every length
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["simpson", "gauss_legendre"])
@pytest.mark.parametrize("d,n", [(1, M - 1), (1, M), (1, M + 63), (2, 511), (2, 513), (2, 723), (2, 725), (3, 63), (3, 65),
                                 (3, 79), (3, 81), (4, 27), (7, 5), (7, 7), (8, 5), (5, 3), (2, 127), (2, 129)])
def test_grid_points_around_the_switch(d, n, rule, dtype, dev):
    dom = _box(d, dtype, dev)
    if rule == "gauss_legendre":
        n = min(n, 20000)
    elif n % 2 == 0:
        n -= 1
    gl = gauss_legendre(n, device=dev) if rule == "gauss_legendre" else None
    pts = _ops.grid_points(_ops.RULES[rule], d, n, dom, gl)
    other = _unaligned(n**d * d, dtype, dev)
    g = _ops.grid_desc(_ops.RULES[rule], d, n, dtype, gl)
    _lib.call("tq_grid_points", ctypes.byref(g), _lib.ptr(dom), _lib.ptr(other), _lib.stream_ptr(dev))
    assert torch.equal(pts, other.view(n**d, d))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("d", [1, 2, 7, 8, 9])
@pytest.mark.parametrize("N", [(1 << 17) - 1, 1 << 17, (1 << 18) - 1, 1 << 18, (1 << 18) + 321])
def test_mc_points_around_the_switch(d, N, dtype, dev):
    dom = torch.tensor([[-0.3, 1.1]] * d, dtype=dtype, device=dev)
    pts = _ops.mc_points(d, N, dom, 77, 5)
    other = _unaligned(N * d, dtype, dev)
    m = _ops.mc_desc(d, N, dtype, 77, 5)
    _lib.call("tq_mc_points", ctypes.byref(m), _lib.ptr(dom), _lib.ptr(other), _lib.stream_ptr(dev))
    assert torch.equal(pts, other.view(N, d))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["boole", "gauss_legendre", "unit"])
@pytest.mark.parametrize("d,n,S", [(1, M - 3, 1), (1, M + 1, 1), (2, 721, 1), (2, 725, 1), (3, 77, 1), (3, 81, 1), (1, 8189, 64),
                                   (1, 8193, 64), (3, 9, 719), (3, 9, 721), (7, 5, 6), (7, 5, 7), (2, 1445, 1), (2, 1449, 1),
                                   (1, 2**20 + 1, 2), (4, 5, 1), (2, 9, 3), (1, 5, 1000)])
def test_reduce_backward_around_the_switch(d, n, S, rule, dtype, dev):
    unit = rule == "unit"
    code = _ops.RULES["gauss_legendre" if unit else rule]
    dom = _box(d, dtype, dev)
    if rule == "boole":
        w, c = np.full(n, 14.0), 1.0 / 22.5 / (n - 1)
        w[1::2], w[2::4], w[0], w[-1] = 32.0, 12.0, 7.0, 7.0
        gl = None
    else:
        w = np.random.default_rng(n).uniform(0.5, 2.0, n)
        gl, c = (torch.linspace(-1.0, 1.0, n, dtype=torch.float64, device=dev), torch.tensor(w, device=dev)), 0.5
        if unit:
            w = np.ones(n)
    g = torch.linspace(-1.0, 2.0, S, dtype=dtype, device=dev)
    gf = _ops.grid_reduce_backward(code, d, n, dom, g, n**d, unit_weights=unit, gl=gl)
    W = torch.prod((dom[:, 1].double() - dom[:, 0].double()) * c).reshape(1)
    for _ in range(d):
        W = (W[:, None] * torch.tensor(w, device=dev)[None, :]).reshape(-1)
    ref = W[:, None] * g.double()[None, :]
    # a product of at most 2 d + 2 FP64 factors, rounded once to the data type
    eps = (2.0**-24 if dtype == torch.float32 else 0.0) + (2 * d + 4) * 2.0**-53
    assert bool(((gf.double() - ref).abs() <= eps * ref.abs()).all())


# one to 257 rows of partials: the final sum's block of 256 and of 1024 threads
@pytest.mark.parametrize("S", [1, 2, 5, 63])
@pytest.mark.parametrize("N", [1, 511, 512, 513, 4096, 100000, 600000])
def test_mean_around_the_final_block(N, S, dev):
    dom = _box(2, torch.float64, dev)
    gen = torch.Generator(device=dev).manual_seed(N + S)
    v = torch.rand((N, S), dtype=torch.float64, device=dev, generator=gen) - 0.25
    vol = float(torch.prod(dom[:, 1] - dom[:, 0]))
    ref = torch.mean(v, dim=0) * vol
    assert float((_ops.mc_reduce(v, dom) - ref).abs().max()) <= vol * (N + 8) * 2.0**-53
