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


# (dim, n, S): one value per load and four, rows that four values cross, one
# axis longer than the weight table, every S class and its edges
VALUES = [(1, 5, 1), (1, 257, 1), (1, 2049, 1), (1, 100001, 1), (2, 45, 1), (2, 49, 1), (3, 101, 1), (5, 9, 1),
          (8, 5, 1), (2, 2501, 1), (3, 9, 2), (2, 33, 3), (4, 5, 31), (2, 65, 63), (1, 2305, 7), (1, 101, 64),
          (2, 17, 65), (1, 10001, 200), (3, 13, 130), (1, 1, 1)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["trapezoid", "boole", "gauss_legendre", "unit"])
@pytest.mark.parametrize("d,n,S", VALUES)
def test_grid_reduce_sizes(d, n, S, rule, dtype, dev):
    unit = rule == "unit"
    if unit:
        rule = "gauss_legendre"
    if rule == "boole":
        n = max(5, n - (n - 1) % 4)
    if rule == "trapezoid":
        n = max(2, n)
    dom = _box(d, dtype, dev, n)
    gl = gauss_legendre(n, device=dev) if rule == "gauss_legendre" else None
    gen = torch.Generator(device=dev).manual_seed(d * 1000 + n + S)
    vals = torch.rand((n**d, S), dtype=dtype, device=dev, generator=gen) - 0.25
    got = _ops.grid_reduce(_ops.RULES[rule], d, n, dom, vals, unit_weights=unit, gl=gl)
    # an unaligned copy takes one value per load
    other = _unaligned(vals.numel(), dtype, dev)
    other.copy_(vals.reshape(-1))
    got2 = _ops.grid_reduce(_ops.RULES[rule], d, n, dom, other.view(n**d, S), unit_weights=unit, gl=gl)
    b = dom.double().cpu().numpy()
    if unit:
        w, scale = np.ones(n), np.prod(0.5 * (b[:, 1] - b[:, 0]))
    elif gl is not None:
        w, scale = gl[1].cpu().numpy(), np.prod(0.5 * (b[:, 1] - b[:, 0]))
    elif rule == "trapezoid":
        w, scale = np.r_[1.0, np.full(n - 2, 2.0), 1.0], np.prod((b[:, 1] - b[:, 0]) / (n - 1) / 2.0)
    else:
        w, scale = np.full(n, 14.0), np.prod((b[:, 1] - b[:, 0]) / (n - 1) / 22.5)
        w[1::2], w[2::4], w[0], w[-1] = 32.0, 12.0, 7.0, 7.0
    W = torch.tensor(w, device=dev)
    full = W
    for _ in range(d - 1):
        full = (full[:, None] * W[None, :]).reshape(-1)
    ref = torch.sum(full[:, None] * vals.double(), dim=0) * scale
    bar = float(torch.max(torch.sum(full[:, None].abs() * vals.double().abs(), dim=0))) * abs(scale)
    # FP64 sums, one rounding of the result; N <= 6.3e6 terms of relative error 2^-53 each, at worst in one direction
    tol = bar * (2.0**-24 if dtype == torch.float32 else 0.0) + bar * vals.shape[0] * 2.0**-53
    assert float((got.double() - ref).abs().max()) <= tol
    assert float((got2.double() - ref).abs().max()) <= tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("N,S", [(1, 1), (255, 1), (1024, 1), (1025, 1), (3000001, 1), (1000, 2), (777, 63), (100, 64),
                                 (4097, 65), (10, 1000)])
def test_mc_reduce_sizes(N, S, dtype, dev):
    dom = _box(3, dtype, dev, N)
    gen = torch.Generator(device=dev).manual_seed(N + S)
    vals = torch.rand((N, S), dtype=dtype, device=dev, generator=gen) - 0.25
    other = _unaligned(vals.numel(), dtype, dev)
    other.copy_(vals.reshape(-1))
    vol = float(torch.prod(dom.double()[:, 1] - dom.double()[:, 0]))
    ref = torch.mean(vals.double(), dim=0) * vol
    tol = vol * ((2.0**-24 if dtype == torch.float32 else 0.0) + N * 2.0**-53)
    for v in (vals, other.view(N, S)):
        assert float((_ops.mc_reduce(v, dom).double() - ref).abs().max()) <= tol


def _axis_weights(rule, n, gl):
    if rule == "gauss_legendre":
        return gl[1].cpu().numpy()
    if rule == "trapezoid":
        return np.r_[1.0, np.full(n - 2, 2.0), 1.0]
    w = np.full(n, 14.0)
    w[1::2], w[2::4], w[0], w[-1] = 32.0, 12.0, 7.0, 7.0
    return w


BACKWARD = [(1, 5, 1), (1, 257, 1), (1, 2049, 1), (1, 30001, 1), (2, 45, 1), (2, 49, 1), (3, 101, 1), (8, 5, 1),
            (2, 301, 1), (2, 2, 1), (3, 9, 2), (2, 33, 3), (4, 5, 31), (1, 1001, 64), (2, 17, 65), (1, 101, 200)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["trapezoid", "boole", "gauss_legendre"])
@pytest.mark.parametrize("d,n,S", BACKWARD)
def test_grid_reduce_vjp_sizes(d, n, S, rule, dtype, dev):
    if rule == "boole":
        n = max(5, n - (n - 1) % 4)
    dom = _box(d, dtype, dev, n)
    gl = gauss_legendre(n, device=dev) if rule == "gauss_legendre" else None
    code = _ops.RULES[rule]
    gen = torch.Generator(device=dev).manual_seed(d * 1000 + n + S)
    g = torch.rand(S, dtype=dtype, device=dev, generator=gen) - 0.25
    out = torch.rand(S, dtype=dtype, device=dev, generator=gen) - 0.25
    gf, gd = _ops.grid_reduce_vjp(code, d, n, dom, g, out, n**d, gl=gl)
    b = dom.double()
    width = b[:, 1] - b[:, 0]
    w = torch.tensor(_axis_weights(rule, n, gl), device=dev)
    c = {"gauss_legendre": 0.5, "trapezoid": 0.5 / (n - 1), "boole": 1.0 / 22.5 / (n - 1)}[rule]
    W = torch.prod(width * c).reshape(1)
    for _ in range(d):
        W = (W[:, None] * w[None, :]).reshape(-1)
    ref = W[:, None] * g.double()[None, :]
    # a product of at most 2 d + 2 FP64 factors, rounded once to the data type
    eps = (2.0**-24 if dtype == torch.float32 else 0.0) + (2 * d + 4) * 2.0**-53
    assert bool(((gf.double() - ref).abs() <= eps * ref.abs()).all())
    other = _unaligned(n**d * S, dtype, dev)
    desc = _ops.grid_desc(code, d, n, dtype, gl)
    _lib.call("tq_grid_reduce_backward", ctypes.byref(desc), _lib.ptr(dom), None, 0, _lib.ptr(g), S, _lib.ptr(other),
              _lib.stream_ptr(dev))
    assert bool(((other.view(n**d, S).double() - ref).abs() <= eps * ref.abs()).all())
    gs = torch.sum(g.double() * out.double())
    bar = float(torch.sum((g.double() * out.double()).abs()))
    rd = torch.stack([-gs / width, gs / width], dim=1)
    tol = bar / width.min() * (S * 2.0**-53) + rd.abs() * eps
    assert bool(((gd.double() - rd).abs() <= tol).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["trapezoid", "gauss_legendre"])
@pytest.mark.parametrize("d,n", [(1, 2), (1, 64), (1, 2049), (1, 40001), (2, 3), (2, 45), (2, 700), (3, 65), (4, 32),
                                 (5, 9), (9, 3), (12, 2)])
def test_grid_points_backward_sizes(d, n, rule, dtype, dev):
    dom = _box(d, dtype, dev, n)
    gl = gauss_legendre(n, device=dev) if rule == "gauss_legendre" else None
    gen = torch.Generator(device=dev).manual_seed(d * 1000 + n)
    gp = torch.rand((n**d, d), dtype=dtype, device=dev, generator=gen) - 0.25
    got = _ops.grid_points_backward(_ops.RULES[rule], d, n, dom, gp, gl).double()
    if gl is None:
        t = torch.arange(n, dtype=torch.float64, device=dev) / (n - 1)
    else:
        t = 0.5 * (1.0 + gl[0])
    g64 = gp.double().view(*([n] * d), d)
    for k in range(d):
        s = g64[..., k].sum(dim=[q for q in range(d) if q != k]) if d > 1 else g64[..., 0]
        gb, ga = torch.sum(s * t), torch.sum(s * (1.0 - t))
        bar = float(gp[:, k].double().abs().sum())
        # FP64 sums of n^d terms, one rounding of the result
        tol = bar * n**d * 2.0**-53 + float(max(ga.abs(), gb.abs())) * (2.0**-24 if dtype == torch.float32 else 0.0)
        assert abs(float(got[k, 0] - ga)) <= tol and abs(float(got[k, 1] - gb)) <= tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("name", ["Trapezoid", "Simpson", "Boole", "GaussLegendre"])
def test_call_gradients_match_recorded_backward(name, dtype, dev):
    """Gradients of a callable's integral with and without a recorded backward
    (create_graph), for the values' and the domain's part."""
    import torchquad_amd as tq

    d, n = 2, 13
    a = torch.tensor([1.3, 0.7], dtype=dtype, device=dev, requires_grad=True)
    dom = _box(d, dtype, dev, 5).requires_grad_()

    def value():
        return getattr(tq, name)().integrate(lambda x: torch.exp(-torch.sum(a * x * x, dim=1)), d, N=n**d,
                                             integration_domain=dom)

    plain = torch.autograd.grad(value(), [a, dom])
    kept = torch.autograd.grad(value(), [a, dom], create_graph=True)
    eps = 2.0**-22 if dtype == torch.float32 else 2.0**-50
    for p, q in zip(plain, kept):
        assert float((p - q).abs().max()) <= eps * float(q.abs().max())
