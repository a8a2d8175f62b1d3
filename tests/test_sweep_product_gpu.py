"""Parameter sweeps from factor tables: values and gradients against FP64
autograd of the separable sums, at the sizes where the plan changes."""
import numpy as np
import pytest
import torch

from torchquad_amd.autograd import gaussian_peak_integrals, oscillatory_integrals, product_peak_integrals
from torchquad_amd.gl_nodes import gauss_legendre

pytestmark = pytest.mark.gpu

# (B, d, n): combined outer lane axes (n <= 16) and one, several lane groups and fewer than a wave, no rows and
# rows, one integral over many blocks, axes longer than a wave, an axis too long for the tables, every dimension
SIZES = [(3, 2, 2), (5, 2, 5), (2, 2, 129), (2, 2, 1001), (1, 2, 4201), (7, 3, 5), (3, 3, 17), (1, 3, 65), (4, 4, 9),
         (9, 4, 32), (1, 4, 45), (3, 5, 5), (2, 5, 13), (2, 6, 5), (2, 7, 5), (2, 8, 3), (70, 3, 9)]


def _nodes(rule, n, dev):
    if rule == "gauss_legendre":
        return gauss_legendre(n, device=dev)
    r = torch.arange(n, dtype=torch.float64, device=dev) * (2.0 / (n - 1)) - 1.0
    w = torch.full((n,), 2.0, dtype=torch.float64, device=dev)
    c = 1.0 / (n - 1)
    if rule == "simpson":
        w[1::2] = 4.0
        c = 2.0 / 3.0 / (n - 1)
    w[0] = w[-1] = 1.0
    return r, w * c


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rule", ["trapezoid", "simpson", "gauss_legendre"])
@pytest.mark.parametrize("fam", ["gaussian", "product", "oscillatory"])
@pytest.mark.parametrize("B,d,n", SIZES)
def test_sweep_product_sizes(B, d, n, fam, rule, dtype, dev, parity):
    if rule == "simpson" and n % 2 == 0:
        n += 1
    rng = np.random.default_rng(1000 * d + n)
    lo = rng.uniform(-1.0, 0.0, (B, d))
    dom = np.stack([lo, lo + rng.uniform(0.5, 1.5, (B, d))], axis=2)

    def leaf(v):
        return torch.tensor(v, dtype=dtype, device=dev).requires_grad_()

    a, dom = leaf(rng.uniform(0.5, 2.0, (B, d))), leaf(dom)
    u = leaf(rng.uniform(-0.1, 0.1, B) if fam == "oscillatory" else rng.uniform(-0.5, 0.5, (B, d)))
    g = torch.tensor(rng.uniform(0.5, 1.5, B), dtype=dtype, device=dev)
    fn = {"gaussian": gaussian_peak_integrals, "product": product_peak_integrals,
          "oscillatory": oscillatory_integrals}[fam]
    val = fn(a, u, dom, n=n, rule=rule)
    got = torch.autograd.grad(val, [a, u, dom], g)

    a6, u6, d6 = (t.detach().double().requires_grad_() for t in (a, u, dom))
    r, w = _nodes(rule, n, dev)
    half = 0.5 * (d6[..., 1] - d6[..., 0])
    x = half[..., None] * r + 0.5 * (d6[..., 1] + d6[..., 0])[..., None]
    if fam == "gaussian":
        f = torch.exp(-((a6[..., None] * (x - u6[..., None])) ** 2))
        ref = torch.prod(half * torch.sum(w * f, dim=2), dim=1)
    elif fam == "product":
        f = 1.0 / (a6[..., None] ** -2 + (x - u6[..., None]) ** 2)
        ref = torch.prod(half * torch.sum(w * f, dim=2), dim=1)
    else:
        f = torch.exp(torch.complex(torch.zeros_like(x), a6[..., None] * x))
        z = torch.prod(half * torch.sum(w * f, dim=2), dim=1)
        ph = 2.0 * np.pi * u6
        ref = torch.cos(ph) * z.real - torch.sin(ph) * z.imag
    want = torch.autograd.grad(ref, [a6, u6, d6], g.double())
    # scale of the sums: sum |W f| per integral (the box's volume for the oscillatory one)
    size = torch.prod(half * 2.0, dim=1).max() if fam == "oscillatory" else ref.abs().max()
    bar = 1e-6 if dtype == torch.float32 else 1e-12  # this package's bars for fused grid rules
    err = float((val.double() - ref).abs().max() / size)
    parity.record(err, bar)
    assert err <= bar
    # every gradient is a sum of W f times factors of at most 2 a^2 |t|, 2 a t^2, 2 pi or 1 / width, within 16 here
    for p, q in zip(got, want):
        err = float((p.double() - q).abs().max() / (16.0 * size))
        parity.record(err, bar)
        assert err <= bar, (fam, rule)
