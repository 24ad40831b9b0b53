"""Volume inner product and dissipation on every group layout of the
wall-normal kernels (4, 6 and 8 coefficients per lane, each at the edges of
its range), against a plain numpy sum over the exact Chebyshev mass matrix.

Bound: a sum of m terms accumulated in any order is within m eps of the sum of
the terms' magnitudes.  A mode's products take at most Ny + 3 Ny additions
and the modes' partials fewer than 64 more; the dissipation's derivative adds
a sum of at most Ny terms to each factor."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


def _mass(Ny):
    n = np.arange(Ny)

    def mu(k):
        even = k % 2 == 0
        return np.where(even, 1.0 / np.where(even, 1.0 - 1.0 * k * k, 1.0), 0.0)
    return 0.5 * (mu(n[:, None] + n[None, :]) + mu(n[:, None] - n[None, :]))


@pytest.mark.parametrize("Ny", [5, 15, 17, 31, 33, 63, 65, 127, 129, 255, 257, 383, 385, 449])
def test_dot_and_dissipation_layouts(gpu, Ny):
    import torch
    cf = gpu
    g = cf.Grid(6, Ny, 5, 2 * np.pi, np.pi)  # even Nx (a Nyquist column), odd Nz
    p = cf.CouetteFlow(g, 1 / 400, 0.01)
    rng = np.random.default_rng(Ny)
    shape = (3,) + g.spec_shape
    decay = (1.0 + np.arange(Ny)[:, None, None]) ** -1.0
    U, V = ((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) * decay for _ in range(2))
    dev = [torch.as_tensor(x, device="cuda") for x in (U, V)]
    w = np.where(np.arange(g.Nxh) == 0, 1.0, 2.0) * (np.arange(g.Nxh) != g.Nx // 2)
    M = _mass(Ny)

    def product(a, b):
        return sum(float((w * (x.conj() * np.tensordot(M, y, 1)).real).sum()) for x, y in zip(a, b))

    def magnitude(a, b):
        return sum(float((w * np.abs(x) * np.tensordot(np.abs(M), np.abs(y), 1)).sum()) for x, y in zip(a, b))

    got = cf.dot(p, dev[0], dev[1])
    assert abs(got - product(U, V)) <= EPS * (4 * Ny + 64) * magnitude(U, V)

    k, n = np.arange(Ny)[:, None], np.arange(Ny)[None, :]
    D = np.where((n > k) & ((n - k) % 2 == 1), np.where(k == 0, n, 2.0 * n), 0.0)
    ik, il = 1j * np.arange(g.Nxh)[None, None, :], 2j * np.array([0, 1, 2, -2, -1])[None, :, None]

    def curl(a, D, ik, il, s):
        dy = lambda f: np.tensordot(D, f, 1)  # noqa: E731
        return [dy(a[2]) + s * il * a[1], il * a[0] + s * ik * a[2], ik * a[1] + s * dy(a[0])]
    W = curl(U, D, ik, il, -1.0)
    A = curl(np.abs(U), D, np.abs(ik), np.abs(il), 1.0)
    got = cf.dissipation_rate(p, dev[0], nu=0.5)
    assert abs(got - 0.5 * product(W, W)) <= 0.5 * EPS * (6 * Ny + 64) * magnitude(A, A)
