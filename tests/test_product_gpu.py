"""The product form of the fused grid rules (integrals of three and more axes)
against FP64 sums of the same rules, at the sizes where its plan changes, and
at parameters where single factors or partial products leave the data type's
range."""
import numpy as np
import pytest
import torch

import torchquad_amd as tq
from torchquad_amd import _ops
from torchquad_amd.gl_nodes import gauss_legendre

pytestmark = pytest.mark.gpu

FAMILIES = ["gaussian_peak", "oscillatory", "product_peak", "exp_linear", "sin_sum", "double_gaussian", "constant"]


def _make(fam, d, seed):
    rng = np.random.default_rng(seed)
    a, u = rng.uniform(0.5, 2.0, d), rng.uniform(-0.5, 0.5, d)
    if fam == "gaussian_peak":
        return tq.GaussianPeak(a, u), [lambda x, k=k: np.exp(-((a[k] * (x - u[k])) ** 2)) for k in range(d)]
    if fam == "product_peak":
        return tq.ProductPeak(a, u), [lambda x, k=k: 1.0 / (a[k] ** -2.0 + (x - u[k]) ** 2) for k in range(d)]
    if fam == "oscillatory":
        w = 0.07
        return tq.Oscillatory(a, w), [
            lambda x, k=k: np.exp(1j * a[k] * x) * (np.exp(2j * np.pi * w) if k == 0 else 1.0) for k in range(d)]
    if fam == "exp_linear":
        return tq.ExpLinear(d, a, 0.3), [lambda x, k=k: np.exp(a[k] * x + (0.3 if k == 0 else 0.0)) for k in range(d)]
    if fam == "sin_sum":
        return tq.SinSum(d, a, u), [lambda x, k=k: np.sin(a[k] * x + u[k]) for k in range(d)]
    if fam == "double_gaussian":
        return tq.DoubleGaussian(d, 0.4), None
    return tq.Constant(d, 1.5), [lambda x: np.ones_like(x)] * d


def _axis(rule, lo, hi, n, gl):
    if rule == "gauss_legendre":
        r, w = gl[0].cpu().numpy(), gl[1].cpu().numpy()
        return 0.5 * (hi - lo) * r + 0.5 * (hi + lo), 0.5 * (hi - lo) * w
    x, h = np.linspace(lo, hi, n), (hi - lo) / (n - 1)
    if rule == "trapezoid":
        w = np.full(n, 2.0)
        c = h / 2.0
    elif rule == "simpson":
        w = np.full(n, 2.0)
        w[1::2], c = 4.0, h / 3.0
    else:
        w = np.full(n, 14.0)
        w[1::2], w[2::4], c = 32.0, 12.0, h / 22.5
    w[0] = w[-1] = 7.0 if rule == "boole" else 1.0
    return x, w * c


def _reference(fam, fn, factors, rule, box, n, gl):
    """(the rule's value, its scale: the sum of |w f|, or an upper bound of it)."""
    axes = [_axis(rule, lo, hi, n, gl) for lo, hi in box]
    if fam == "sin_sum":
        s = [np.sum(w * f(x)) for (x, w), f in zip(axes, factors)]
        t = [np.sum(w) for _, w in axes]
        v = sum(s[k] * np.prod(t[:k] + t[k + 1:]) for k in range(len(s)))
        return v, len(s) * np.prod(t)
    if fam == "double_gaussian":
        width, norm = 0.4, 0.5 * (0.4 * np.sqrt(np.pi)) ** -len(box)
        v = norm * sum(np.prod([np.sum(w * np.exp(-((x - c) / width) ** 2)) for x, w in axes]) for c in fn.centers)
        return v, v
    p = np.prod([np.sum(w * f(x)) for (x, w), f in zip(axes, factors)])
    if fam == "oscillatory":
        return p.real, np.prod([np.sum(w) for _, w in axes])
    if fam == "constant":
        p = 1.5 * p
    return p, abs(p)


# (dim, n): the smallest axes; the lane-, wave- and block-built tables (64, 128); one and two loop axes;
# 2, 4 and 8 states per lane (8.4e6, 3.4e7 and 1.3e8 points); many axes
SIZES = [(3, 5), (3, 9), (3, 65), (3, 101), (3, 125), (3, 129), (4, 33), (3, 205), (4, 77), (5, 45), (6, 5), (9, 5)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["trapezoid", "simpson", "boole", "gauss_legendre"])
@pytest.mark.parametrize("d,n", SIZES)
def test_product_sizes(d, n, rule, dtype, dev, parity):
    gl = gauss_legendre(n, device=dev) if rule == "gauss_legendre" else None
    bar = 1e-6 if dtype == torch.float32 else 1e-12  # this package's bars for fused grid rules
    for fam in FAMILIES:
        fn, factors = _make(fam, d, 10 * d + n)
        dom = torch.tensor([[-0.75, 1.25], [-1.0, 0.5]] * 8, dtype=dtype, device=dev)[:d].contiguous()
        got = float(_ops.grid_integrate(_ops.RULES[rule], fn, d, n, dom, gl))
        ref, scale = _reference(fam, fn, factors, rule, dom.double().cpu().numpy(), n, gl)
        parity.record(abs(got - ref) / scale, bar)
        assert abs(got - ref) <= bar * scale, (fam, got, ref)


@pytest.mark.parametrize("ipw,lanes", [(1, 0), (5, 0), (64, 1), (1000, 2), (0, 1), (0, 3), (10**9, 0)])
def test_product_geometry_overrides(ipw, lanes, dev):
    """Any lane axes and items per wave give the same integral."""
    fn, factors = _make("gaussian_peak", 4, 3)
    dom = torch.tensor([[-1.0, 1.0]] * 4, dtype=torch.float64, device=dev)
    ref, _ = _reference("gaussian_peak", fn, factors, "boole", [(-1.0, 1.0)] * 4, 13, None)
    got = float(_ops.grid_integrate(_ops.RULES["boole"], fn, 4, 13, dom, lane_axes=lanes, items_per_wave=ipw))
    assert abs(got - ref) <= 1e-12 * ref


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_factors_outside_the_range(dtype, dev):
    """Single factors that overflow or vanish while the integral is an
    ordinary number, and integrals that are infinite."""
    f32 = dtype == torch.float32
    dom = torch.tensor([[0.0, 1.0]] * 4, dtype=dtype, device=dev)
    rule = _ops.RULES["boole"]
    one = [(0.0, 1.0)]

    def value(fn, n=17):
        return float(_ops.grid_integrate(rule, fn, 4, n, dom))

    def axis_sum(f, n=17):
        x, w = _axis("boole", 0.0, 1.0, n, None)
        return np.sum(w * f(x))

    # e^(80 x) e^(-80 x) ... : the product of the first two axes' sums is e^80/80^2
    a = np.array([80.0, -80.0, 60.0, -60.0]) if f32 else np.array([900.0, -900.0, 300.0, -300.0]) * 0.7
    ref = np.prod([axis_sum(lambda x, k=k: np.exp(a[k] * x - max(a[k], 0.0))) for k in range(4)])
    ref *= np.exp(np.sum(np.maximum(a, 0.0)) - 138.0) if f32 else np.exp(np.sum(np.maximum(a, 0.0)) - 800.0)
    got = value(tq.ExpLinear(4, a, -138.0 if f32 else -800.0))
    # exponents of up to 140 (FP64: 800) octaves carry the rounding of the parameters
    assert abs(got - ref) <= (280 * 2.0**-23 if f32 else 1600 * 2.0**-51) * ref
    # a peak far outside the box: e^-75 (FP64: e^-600) at the nearest corner
    s = 2.5 if f32 else 7.0
    ref = axis_sum(lambda x: np.exp(-((s * (x - 2.7)) ** 2))) ** 4
    got = value(tq.GaussianPeak([s] * 4, [2.7] * 4))
    assert abs(got - ref) <= (4 * 46 * 2.0**-21 if f32 else 4 * 360 * 2.0**-50) * ref
    # product peaks whose factors are 1e+-12 each in turn
    ref = np.prod([axis_sum(lambda x, k=k: 1.0 / (c**-2.0 + (x - 0.5) ** 2)) for k, c in enumerate([1e6, 1e-6, 1e6, 1e-6])])
    got = value(tq.ProductPeak([1e6, 1e-6, 1e6, 1e-6], [0.5] * 4))
    assert abs(got - ref) <= (1e-6 if f32 else 1e-12) * ref
    # an integral beyond the type, a singular peak on a node (0 * inf in the sum), NaN parameters
    assert value(tq.ExpLinear(4, [400.0] * 4 if f32 else [4000.0] * 4)) == float("inf")
    assert np.isnan(value(tq.ProductPeak([1e30] * 4 if f32 else [1e200] * 4, [0.5] * 4)))
    assert np.isnan(value(tq.GaussianPeak([1.0, float("nan"), 1.0, 1.0], [0.0] * 4)))


def test_product_custom_weights(dev):
    """A Gaussian rule whose weights span 80 orders of magnitude and one with negative weights."""
    import scipy.special

    x, w = scipy.special.roots_hermite(101)
    gl = (torch.tensor(x, device=dev), torch.tensor(w, device=dev))
    dom = torch.tensor([[-1.0, 1.0]] * 3, dtype=torch.float64, device=dev)
    got = float(_ops.grid_integrate(_ops.RULES["gauss_legendre"], tq.ExpLinear(3, [1.0, 2.0, -1.5]), 3, 101, dom, gl))
    ref = np.pi**1.5 * np.exp((1.0 + 4.0 + 2.25) / 4.0)  # integral of e^(-x^2 + a x) per axis
    assert abs(got - ref) <= 1e-12 * ref
    r = np.array([-0.5, 0.0, 0.75, 0.9])
    wn = np.array([0.5, -0.25, 1.0, 0.75])
    gl = (torch.tensor(r, device=dev), torch.tensor(wn, device=dev))
    for dtype, bar in ((torch.float32, 1e-6), (torch.float64, 1e-12)):
        got = float(_ops.grid_integrate(_ops.RULES["gauss_legendre"], tq.GaussianPeak([1.0] * 3, [0.25] * 3), 3, 4,
                                        dom.to(dtype), gl))
        per_axis = np.sum(wn * np.exp(-((r - 0.25) ** 2)))
        scale = np.sum(np.abs(wn) * np.exp(-((r - 0.25) ** 2))) ** 3
        assert abs(got - per_axis**3) <= bar * scale


def _batch_item(rule, fam, d, n, seed):
    fn, factors = _make(fam, d, seed)
    return {"rule": rule, "fn": fn, "dim": d, "n": n, "domain": [[-0.75, 1.25], [-1.0, 0.5]] * (d // 2)
            + [[-0.75, 1.25]] * (d % 2)}, factors


# (dim, n): two axes, table classes (26 and 60 KB), axes too long for them, one and two loop axes (n = 32, 33),
# more lane groups than tiles, more tiles than lane groups, no full lane group, rows
BATCH = [(2, 2), (2, 33), (2, 129), (2, 701), (2, 2301), (3, 2), (3, 21), (3, 32), (3, 33), (3, 101), (4, 5), (4, 31),
         (5, 9), (6, 10), (7, 3), (8, 5)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["trapezoid", "simpson", "gauss_legendre"])
@pytest.mark.parametrize("tile_points", [64, 8192, 1 << 20])
def test_batch_product_sizes(tile_points, rule, dtype, dev, parity):
    """Every family at every size in one batch, with classes and (the same
    tiles on the general kernel) without."""
    from torchquad_amd import _lib
    from torchquad_amd.batch import Batch

    specs = []
    for d, n in BATCH:
        if tile_points == 64 and n**d > 2e5:
            continue  # tens of thousands of tiles say nothing new
        if rule == "simpson" and n % 2 == 0:
            n += 1
        for fam in FAMILIES:
            specs.append((fam, d, n, *_batch_item(rule, fam, d, n, 31 * d + n)))
    b = Batch([s[3] for s in specs], dtype=dtype, device=dev, tile_points=tile_points)
    out64 = b.run()[1].clone()
    alone = torch.empty_like(out64)
    _lib.call("tq_batch_run", b.dt, _lib.ptr(b.desc), b.count, _lib.ptr(b.tiles), b.n_tiles, _lib.ptr(b.tile_begin),
              _lib.ptr(b.tile_count), _lib.ptr(b.gl_x), _lib.ptr(b.gl_w), _lib.ptr(b.gl_p32),
              b.gl_x.numel() if b.gl_x is not None else 0, _lib.ptr(b.tile_part), None, _lib.ptr(alone), None,
              _lib.stream_ptr(dev))
    bar = 1e-6 if dtype == torch.float32 else 1e-12
    for i, (fam, d, n, item, factors) in enumerate(specs):
        gl = gauss_legendre(n, device=dev) if rule == "gauss_legendre" else None
        ref, scale = _reference(fam, item["fn"], factors, rule, item["domain"], n, gl)
        for v in (float(out64[i]), float(alone[i])):
            parity.record(abs(v - ref) / scale, bar)
            assert abs(v - ref) <= bar * scale, (fam, d, n, v, ref)
