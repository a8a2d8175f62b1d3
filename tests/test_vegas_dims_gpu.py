"""VEGAS sampling at the edges of its dimension classes (4 | 6 | 8 | 16): the
fused kernel against the point writer with the map and sums of user values."""
import warnings

import pytest
import torch

import torchquad_amd as tq

pytestmark = pytest.mark.gpu


# Both draw the same stream.  FP32 values of cos at arguments up to 30 rad differ by 4e-6 at most
# (in units of the volume), FP64 ones by 1e-14; the sums' order (atomics for wide maps) adds less.
# Not a constant: its variances are rounding noise, which the stratification would follow.
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 4e-6), (torch.float64, 1e-11)])
@pytest.mark.parametrize("d,N", [(1, 1500), (2, 4097), (4, 30011), (5, 30011), (6, 50021), (7, 30011), (8, 40009),
                                 (9, 30011), (12, 20011)])
def test_fused_and_point_sampling_agree(d, N, dtype, tol, dev):
    dom = torch.tensor([[0.0, 1.0 + 0.25 * k] for k in range(d)], dtype=dtype, device=dev)
    f = tq.Oscillatory([1.0 + 0.1 * k for k in range(d)], 0.1)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        fused = float(tq.VEGAS().integrate(f, d, N=N, integration_domain=dom, seed=5))
        user = float(tq.VEGAS().integrate(lambda x: f(x), d, N=N, integration_domain=dom, seed=5))
    volume = float((dom[:, 1] - dom[:, 0]).cpu().double().prod())
    assert abs(fused - user) <= tol * volume
