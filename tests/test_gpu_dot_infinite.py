"""The inner product of a field with an infinite coefficient is the infinity
that its terms sum to: the degrees that pad a lane group's columns past Ny
take no part.  One entry per group layout, Ny below and at its full width."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("Ny", [5, 15, 17, 31, 33, 97, 129, 255, 257, 383, 385, 511])
def test_dot_with_an_infinite_coefficient(gpu, Ny, sign):
    import torch
    cf = gpu
    g = cf.Grid(6, Ny, 5, 2 * np.pi, np.pi)
    p = cf.CouetteFlow(g, 1 / 400, 0.01)
    U = np.zeros((3,) + g.spec_shape, dtype=complex)
    V = np.zeros_like(U)
    U[0, :, 0, 0] = -1.0  # the products M_m0 v_0, M_m0 = 1 / (1 - m^2) for even m, all have the sign of v_0
    U[0, 0, 0, 0] = 1.0
    V[0, 0, 0, 0] = sign * np.inf
    dev = [torch.as_tensor(x, device="cuda") for x in (U, V)]
    assert cf.dot(p, *dev) == sign * np.inf
