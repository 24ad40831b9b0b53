"""A velocity component that is identically zero stays zero bit for bit.

In two dimensions (no variation in z, V_z = 0) every product of the spanwise
equation has a factor that is exactly zero, so V_z, and whatever the passes
make of a zero field, holds zeros: the transforms are linear and no field's
rounding errors may enter another.  Streamwise padded lengths: even and odd,
each of the small radices of the x pass, and lengths that it does not split."""
import numpy as np
import pytest

from test_gpu_parity import hermitian_random, make

pytestmark = pytest.mark.gpu

# padded x lengths 6, 9, 12, 18, 25, 33, 36, 45, 48, 51, 54, 63, 81, 96, 120, 150, 192, 288, 384
NX = [4, 6, 8, 12, 17, 22, 24, 30, 32, 34, 36, 42, 54, 64, 80, 100, 128, 192, 256]


def _plane_state(go, rng):
    U = hermitian_random(go, rng, 3) * 0.1
    U[:, :, 1:] = 0.0  # l = 0 alone
    U[2] = 0.0
    return U


@pytest.mark.parametrize("form", ["rotating", "convective", "divergence"])
@pytest.mark.parametrize("Nx", NX)
def test_zero_component_stays_zero(gpu, Nx, form):
    import torch
    cf = gpu
    gc, go, prob = make(cf, (Nx, 9, 6), form=form)
    rng = np.random.default_rng(Nx)
    U = torch.as_tensor(_plane_state(go, rng), device="cuda")
    N = prob.nlterm(0.0, U)
    assert N[0].abs().max() > 0 and N[2].abs().max() == 0
    cf.project_(U, prob)
    P = cf.pressure(U, prob)
    cf.step_(prob.scheme, prob.nlterm, U, P, 0.0, nsteps=2, **prob.constraint)
    assert U[0].abs().max() > 0 and U[2].abs().max() == 0


@pytest.mark.parametrize("Nx", [n for n in NX if (3 * n + 1) // 2 % 2 == 0])  # velocity_gradient takes even padded lengths
def test_zero_derivatives(gpu, Nx):
    import torch
    cf = gpu
    gc, go, prob = make(cf, (Nx, 9, 6))
    U = torch.as_tensor(_plane_state(go, np.random.default_rng(Nx)), device="cuda")
    g = cf.velocity_gradient(prob, U)
    assert g[0, 1].abs().max() > 0
    assert g[2].abs().max() == 0 and g[:, 2].abs().max() == 0  # dV_z/dx_j, dV_i/dz
