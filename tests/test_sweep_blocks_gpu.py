"""Sweeps whose integrals differ by many orders of magnitude, at the sizes where
the number of waves per block changes: every integral and every one of its
gradients is held against its own size."""
import numpy as np
import pytest
import torch

from torchquad_amd.autograd import gaussian_peak_integrals, product_peak_integrals

pytestmark = pytest.mark.gpu


# 1024, 2048 and 4096 points per integral and their neighbours; one block, several blocks, all of eight waves
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("fam", ["gaussian", "product"])
@pytest.mark.parametrize("B,d,n", [(9, 2, 31), (9, 2, 33), (9, 3, 11), (5, 2, 45), (5, 2, 47), (5, 3, 13), (5, 4, 7), (5, 2, 63),
                                   (5, 2, 65), (3, 4, 9), (3, 5, 5), (2, 3, 61), (40, 6, 3), (4, 8, 3)])
def test_every_integral_by_its_own_size(B, d, n, fam, dtype, dev, parity):
    rng = np.random.default_rng(100 * d + n)
    lo = rng.uniform(-1.0, 0.0, (B, d))
    dom = np.stack([lo, lo + rng.uniform(0.5, 1.5, (B, d))], axis=2)
    a = rng.uniform(0.5, 2.0, (B, d))
    u = rng.uniform(-2.0, 2.0, (B, d)) if fam == "gaussian" else rng.uniform(-30.0, 30.0, (B, d))

    def leaf(v):
        return torch.tensor(v, dtype=dtype, device=dev).requires_grad_()

    a, u, dom = leaf(a), leaf(u), leaf(dom)
    fn = gaussian_peak_integrals if fam == "gaussian" else product_peak_integrals
    val = fn(a, u, dom, n=n, rule="simpson")
    got = torch.autograd.grad(val.sum(), [a, u, dom])

    a6, u6, d6 = (t.detach().double().requires_grad_() for t in (a, u, dom))
    r = torch.arange(n, dtype=torch.float64, device=dev) * (2.0 / (n - 1)) - 1.0
    w = torch.full((n,), 2.0, dtype=torch.float64, device=dev)
    w[1::2] = 4.0
    w[0] = w[-1] = 1.0
    w *= 2.0 / 3.0 / (n - 1)
    half = 0.5 * (d6[..., 1] - d6[..., 0])
    x = half[..., None] * r + 0.5 * (d6[..., 1] + d6[..., 0])[..., None]
    t = x - u6[..., None]
    f = torch.exp(-((a6[..., None] * t) ** 2)) if fam == "gaussian" else 1.0 / (a6[..., None] ** -2 + t**2)
    ref = torch.prod(half * torch.sum(w * f, dim=2), dim=1)
    want = torch.autograd.grad(ref.sum(), [a6, u6, d6])
    eps = 2.0**-23 if dtype == torch.float32 else 2.0**-52
    # a value: d factors of a few roundings each; the rounding of a and a u enters the exponents, which reach
    # `octaves` over the box, twice.  x and u are of size 30 at most, distances of size 28 to 31 lose five bits.
    with torch.no_grad():
        octaves = 2.0 * torch.sum(torch.amax((a6[..., None] * t) ** 2, dim=2), dim=1) if fam == "gaussian" else 32.0
        size = ref.abs()
        bar = (4 * d + 2 * octaves) * eps
        err = (val.double() - ref).abs() / size / bar
        parity.record(float(err.max()), 1.0)
        assert bool((err <= 1.0).all())
        # a gradient: W f times 2 a^2 |t|, 2 a t^2 (product: 2 |t g|, 2 g / a^3) or 1 / width and those, each at its largest
        tm = torch.amax(t.abs(), dim=2)
        if fam == "gaussian":
            ga, gu = 2.0 * a6 * tm**2, 2.0 * a6**2 * tm
        else:
            gm = torch.amax(f, dim=2)
            ga, gu = 2.0 * gm / a6**3, 2.0 * tm * gm
        scale = [ga, gu, (gu + 1.0 / (2.0 * half))[..., None].expand(-1, -1, 2)]
        for p, q, s in zip(got, want, scale):
            b = (bar * size).reshape(-1, *[1] * (s.dim() - 1)) * s
            err = (p.double() - q).abs() / b
            parity.record(float(err.max()), 1.0)
            assert bool((err <= 1.0).all())
