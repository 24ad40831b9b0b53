"""Periodic passes at the edges of their length rules: lines kept in one lane,
each pair of register radices, lengths with no such pair (the staged passes),
widths that do not divide the tile.  Transforms against the oracle, at the flat
1e-13 that every transform of the repository is held to; the nonlinear step
against the oracle's step within its roundoff envelope."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_parity import _split, assert_parity, hermitian_random, make, rel, run_pair, say

pytestmark = pytest.mark.gpu

# padded z lengths 2, 3, 11, 12, 14, 21, 24, 48, 50, 98, 105, 192, 225, 288, 360, 384, 432, 504, 576, 600
NZ = [1, 2, 7, 8, 9, 14, 16, 32, 33, 65, 70, 128, 150, 192, 240, 256, 288, 336, 384, 400]


@pytest.mark.parametrize("Nz", NZ)
@pytest.mark.parametrize("Nx", [5, 12, 34])
def test_z_lengths(gpu, Nz, Nx):
    import torch
    cf = gpu
    say("z length", Nx, Nz)
    gc, go, prob = make(cf, (Nx, 5, Nz))
    rng = np.random.default_rng(Nz + 1000 * Nx)
    u = rng.standard_normal((3,) + go.phys_shape)
    F = cf.FFT(prob, torch.as_tensor(u, device="cuda")).cpu().numpy()
    U = hermitian_random(go, rng, 3)
    v = cf.IFFT(prob, torch.as_tensor(U, device="cuda")).cpu().numpy()
    for c in range(3):
        assert rel(F[c], O.forward(go, u[c])) < 1e-13
        assert rel(v[c], O.inverse(go, U[c])) < 1e-13


# padded x lengths 2, 3, 5, 6, 8, 9, 11, 12, 14, 21, 33 and 51 (odd, 51 staged), 63, 81, 98 .. 384: each register
# class of the x pass, the shortest lines, odd and even, and lengths that keep the staged pass
NX = [1, 2, 3, 4, 5, 6, 7, 8, 9, 14, 22, 34, 42, 54, 65, 70, 96, 128, 150, 160, 192, 200, 256, 300]


@pytest.mark.parametrize("Nx", NX)
def test_x_lengths(gpu, Nx):
    import torch
    cf = gpu
    say("x length", Nx)
    gc, go, prob = make(cf, (Nx, 5, 6))
    rng = np.random.default_rng(Nx)
    u = rng.standard_normal((3,) + go.phys_shape)
    F = cf.FFT(prob, torch.as_tensor(u, device="cuda")).cpu().numpy()
    U = hermitian_random(go, rng, 3)
    v = cf.IFFT(prob, torch.as_tensor(U, device="cuda")).cpu().numpy()
    for c in range(3):
        assert rel(F[c], O.forward(go, u[c])) < 1e-13
        assert rel(v[c], O.inverse(go, U[c])) < 1e-13


@pytest.mark.parametrize("form", ["rotating", "convective", "divergence"])
@pytest.mark.parametrize("Nx", [3, 4, 5, 8, 14, 30, 42, 64, 65, 100, 150, 200, 256])
def test_x_lengths_step(gpu, Nx, form):
    say("x length step", form, Nx)
    U, P, Ur, Pr, _, _, env = run_pair(gpu, (Nx, 9, 6), 1, form=form)
    assert_parity(f"step {form} {Nx}", _split((U, P)), _split((Ur, Pr)), env)


# each pair of register radices of the wall-normal transform (2 x 4 .. 24 x 24, 16 x 32), one to three fields a
# pass, the edges of the lane layouts, and a length that keeps the staged transform (197)
NY = [5, 7, 9, 13, 17, 19, 21, 25, 29, 31, 33, 37, 43, 49, 51, 57, 61, 65, 73, 81, 85, 91, 97, 101, 109, 113, 121, 127,
      129, 141, 145, 151, 161, 163, 181, 193, 197, 211, 241, 253, 257, 289, 321, 337]


@pytest.mark.parametrize("Ny", NY)
def test_y_lengths_step(gpu, Ny):
    say("y length step", Ny)
    U, P, Ur, Pr, _, _, env = run_pair(gpu, (8, Ny, 7), 1)
    assert_parity(f"step {Ny}", _split((U, P)), _split((Ur, Pr)), env)


@pytest.mark.parametrize("form", ["convective", "divergence"])
@pytest.mark.parametrize("Ny", [9, 17, 33, 49, 65, 97, 101, 129, 193, 257])
def test_y_lengths_forms(gpu, Ny, form):
    say("y length form", form, Ny)
    U, P, Ur, Pr, _, _, env = run_pair(gpu, (7, Ny, 8), 1, form=form)
    assert_parity(f"step {form} {Ny}", _split((U, P)), _split((Ur, Pr)), env)
