"""Hooks of the grid integrators on the user-callable path."""
import pytest
import torch

import torchquad_amd as tq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,N", [("Trapezoid", 25), ("Simpson", 25), ("GaussLegendre", 16)])
def test_calculate_grid_set_on_the_instance(name, N, dev):
    """calculate_grid may be replaced on one object as well as by a subclass."""
    integ = getattr(tq, name)()
    dom = torch.tensor([[0.0, 1.0], [0.0, 2.0]], dtype=torch.float64, device=dev)
    plain = integ.integrate(lambda x: x[:, 0] * x[:, 1], 2, N=N, integration_domain=dom)
    own, calls = integ.calculate_grid, []

    def calculate_grid(*args, **kwargs):
        calls.append(args)
        return own(*args, **kwargs)

    integ.calculate_grid = calculate_grid
    value = integ.integrate(lambda x: x[:, 0] * x[:, 1], 2, N=N, integration_domain=dom)
    assert len(calls) == 1
    assert abs(float(value - plain)) <= 1e-14 * abs(float(plain))
