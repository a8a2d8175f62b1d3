"""The Monte Carlo kernel of every dimension: a counter that passes 2^32 inside
one thread's run, and an axis whose size times 2^-24 leaves the normal range."""
import pytest
import torch

import torchquad_amd as tq
from torchquad_amd import _ops

pytestmark = pytest.mark.gpu


# |exponent| <= 4.5: 18 roundings of at most 6.5 (in units of log2) in the
# exponent and 32 sums of positive values give 7e-6 in FP32, 2e-14 in FP64
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.float64, 1e-13)])
@pytest.mark.parametrize("size", [1.5, 1e-33])
@pytest.mark.parametrize("d", range(1, 17))
def test_sums_against_the_stream_points(d, size, dtype, tol, dev):
    N, seed, offset = 5003, 11, 2**32 - 1000
    dom = torch.tensor([[0.0, size]] + [[-0.5, 1.0]] * (d - 1), dtype=dtype, device=dev)
    a = torch.tensor([3.0 / size] + [0.1] * (d - 1), dtype=torch.float64)
    f = tq.ExpLinear(d, a=a.tolist())
    stats = torch.zeros(3, dtype=torch.float64, device=dev)
    _ops.mc_integrate(f, d, N, dom, seed, offset=offset, stats=stats, samples_per_thread=33)
    x = _ops.mc_points(d, N, dom, seed, offset=offset).cpu().double()
    y = torch.exp((x * a.to(dtype).double()).sum(1))
    width = dom.cpu().double()
    vol = float((width[:, 1] - width[:, 0]).prod())
    got = stats.cpu()
    assert abs(float(got[0]) / (vol * float(y.sum())) - 1) <= tol
    assert abs(float(got[1]) / (vol * vol * float((y * y).sum())) - 1) <= 2 * tol
    assert float(got[2]) == N
