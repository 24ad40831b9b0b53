"""The public nonlinear term is the step's own, and as accurate as plain FP64
sums, over the streamwise padded lengths.

Identity: a forcing of minus the nonlinear term cancels the step's exactly if
both come out of the same passes, and leaves the linear step.  That step is
also what fields scaled by 2^-600 take, whose products (2^-1200) are zero in
FP64 while every linear operation scales exactly by a power of two.  The
divergence form assembles its term in one kernel for both callers, so the
comparison is bit for bit.

Accuracy: each component's rms distance from the extended-precision oracle
against the FP64 oracle's.  Both are sums over the same terms with about the
same number of roundings, so their error variances are alike; sqrt(2) allows
twice the variance."""
import math

import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_parity import hermitian_random, make, rel, say

pytestmark = pytest.mark.gpu


# padded lengths 9, 24, 48, 51, 81, 192, 288
@pytest.mark.parametrize("Nx", [6, 16, 32, 34, 54, 128, 192])
def test_forcing_by_minus_the_nonlinear_term_cancels_it(gpu, Nx):
    import torch
    cf = gpu
    dims = (Nx, 9, 6)
    gc, go, prob = make(cf, dims, profile=lambda y: 0.0 * y, form="divergence")
    _, _, other = make(cf, dims, profile=lambda y: 0.0 * y, form="divergence")  # the callback's own workspace
    U0 = torch.as_tensor(0.1 * hermitian_random(go, np.random.default_rng(Nx), 3), device="cuda")
    cf.project_(U0, prob)
    P0 = cf.pressure(U0, prob)

    def cancel(t, U, F):
        F -= other.nlterm(t, U)

    U, P = U0.clone(), P0.clone()
    cf.step_(prob.scheme, prob.nlterm, U, P, 0.0, forcing=cancel, **prob.constraint)
    s = 2.0 ** -600
    V, Q = U0 * s, P0 * s
    cf.step_(prob.scheme, prob.nlterm, V, Q, 0.0, **prob.constraint)
    assert U.abs().max() > 0
    assert torch.equal(U, V / s) and torch.equal(P, Q / s)


# padded lengths whose second radix is 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 15, 16, and 33, 51, 66 (staged)
@pytest.mark.parametrize("form", ["rotating", "convective", "divergence"])
@pytest.mark.parametrize("Nx", [8, 16, 24, 40, 64, 42, 128, 54, 100, 192, 150, 256, 22, 34, 44])
def test_nonlinear_lengths(gpu, Nx, form):
    import torch
    cf = gpu
    gc, go, prob = make(cf, (Nx, 9, 6), form=form)
    U = hermitian_random(go, np.random.default_rng(Nx), 3)
    N = prob.nlterm(0.0, torch.as_tensor(U, device="cuda")).cpu().numpy()
    Nr = O.Problem(go, lambda y: y, 1 / 400, 0.01, form=form).nonlinear(U)
    say(f"nonlinear {form} Nx {Nx}: {rel(N, Nr):.3e}")
    assert rel(N, Nr) < 1e-12


# of these lengths the even ones, which velocity_gradient takes
@pytest.mark.parametrize("Nx", [8, 16, 24, 40, 64, 128, 100, 192, 256, 44])
def test_velocity_gradient_lengths(gpu, Nx):
    import torch
    cf = gpu
    gc, go, prob = make(cf, (Nx, 9, 6))
    U = hermitian_random(go, np.random.default_rng(Nx), 3)
    got = cf.velocity_gradient(prob, torch.as_tensor(U, device="cuda")).cpu().numpy()
    U[0, 1, 0, 0] += 1.0  # the base flow y = T_1
    for i in range(3):
        for j, op in enumerate(("ddx1", "ddx2", "ddx3")):
            assert rel(got[i, j], O.inverse(go, O.operator(go, op, U[i]))) < 1e-12, (i, j)


def test_nonlinear_accuracy_by_component(gpu):
    """Plane Poiseuille at 64x65x64, four perturbed states, geometric mean."""
    cf = gpu
    dims, box = (64, 65, 64), (4 * math.pi, 4 * math.pi / 3)
    prof = lambda y: 1.5 * (1 - y ** 2)  # noqa: E731
    gc, go, prob = make(cf, dims, box, profile=prof, nu=1 / 2800, dt=0.005, bulkvelocity=(1.0, 0.0))
    ref = O.Problem(go, prof, 1 / 2800, 0.005, bulkvelocity=(1.0, 0.0))
    ext = O.Problem(go, prof, 1 / 2800, 0.005, bulkvelocity=(1.0, 0.0), extended=True)
    logs = np.zeros(3)
    for seed in range(4):
        U = cf.perturbation_state(prob, 0.05, seed=seed).velocity
        N = prob.nlterm(0.0, U).cpu().numpy()
        Uh = U.cpu().numpy()
        X, R = ext.nonlinear(Uh), ref.nonlinear(Uh)
        rms = lambda a: np.sqrt((np.abs(a - X) ** 2).mean(axis=(1, 2, 3)))  # noqa: E731
        logs += np.log(rms(N) / rms(R)) / 4
    say(f"nonlinear term, rms error over the oracle's: {np.exp(logs)}")
    assert (np.exp(logs) < math.sqrt(2)).all(), np.exp(logs)
