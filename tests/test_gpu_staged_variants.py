"""The staged x pass of the FP64 fields, where it still runs: every variant and
wavefront count gives the same bits, in the step of padded lengths without
register radices and in pressure; and transforms() tells which transforms a
step runs."""
import math

import numpy as np
import pytest

from test_gpu_parity import _split, assert_parity, run_pair, say

pytestmark = pytest.mark.gpu
BOX = (2 * math.pi, math.pi)


def _problem(cf, dims, **kw):
    return cf.ChannelFlowProblem(cf.Grid(*dims, *BOX), lambda y: 1.5 * (1 - y ** 2), 1 / 2800, 0.002,
                                 bulkvelocity=(1.0, 0.0), **kw)


def _choices(cf, prob):
    """(x variant, waves) choices the problem accepts, the default one first."""
    keep = cf.get_tiles(prob)
    out = [(keep[2], keep[3])]
    for var in (0, 1, 2):
        for w in (1, 2, 3, 4):
            try:
                cf.set_tiles(prob, keep[0], var, w)
            except ValueError:
                continue
            out.append((var, w))
    cf.set_tiles(prob, keep[0], keep[2], keep[3])
    return keep[0], out


# padded Nx 66 (a radix 11: two buffers), 324 (all three variants), 450, 576: even, without register radices
@pytest.mark.parametrize("Nx", [44, 216, 300, 384])
def test_step_of_unsplit_lengths(gpu, Nx):
    import torch
    cf = gpu
    prob = _problem(cf, (Nx, 9, 6))
    assert cf.transforms(prob)["x"] == (0, 0)
    st = cf.perturbation_state(prob, 0.05, seed=Nx)
    kt, choices = _choices(cf, prob)
    assert Nx != 216 or {v for v, _ in choices} == {0, 1, 2}
    first = None
    for var, w in choices:
        cf.set_tiles(prob, kt, var, w)
        U, P = st.velocity.clone(), st.stagepressure.clone()
        cf.step_(prob.scheme, prob.nlterm, U, P, 0.0, nsteps=2, **prob.constraint)
        if first is None:
            first = U, P
        assert torch.equal(U, first[0]) and torch.equal(P, first[1]), (var, w)


@pytest.mark.parametrize("Nx", [216, 384])
def test_step_of_unsplit_lengths_against_the_oracle(gpu, Nx):
    say("unsplit length", Nx)
    U, P, Ur, Pr, _, _, env = run_pair(gpu, (Nx, 9, 6), 1)
    assert_parity(f"step {Nx}", _split((U, P)), _split((Ur, Pr)), env)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("Nx", [16, 32, 128])
def test_pressure_of_split_lengths(gpu, Nx, precision):
    import torch
    cf = gpu
    prob = _problem(cf, (Nx, 17, 8), precision=precision)
    U = cf.perturbation_state(prob, 0.05, seed=Nx).velocity
    kt, choices = _choices(cf, prob)
    assert {v for v, _ in choices} == {0, 1, 2}
    first = None
    for var, w in choices:
        cf.set_tiles(prob, kt, var, w)
        P = cf.pressure(U, prob)
        if first is None:
            first = P
        assert torch.equal(P, first), (var, w)


def test_transforms_report(gpu):
    cf = gpu
    prob = _problem(cf, (128, 97, 128))
    assert cf.transforms(prob) == {"x": (24, 8), "z": (16, 12), "y": (12, 16)}
    keep = cf.get_tiles(prob)
    cf.set_tiles(prob, keep[0], keep[2], keep[3], y_coefs=8)  # a layout with the staged transform
    assert cf.transforms(prob) == {"x": (24, 8), "z": (16, 12), "y": (0, 0)}
    assert cf.transforms(_problem(cf, (22, 197, 8))) == {"x": (0, 0), "z": (12, 1), "y": (0, 0)}
    assert cf.transforms(_problem(cf, (32, 33, 32), precision="mixed")) == {"x": (0, 0), "z": (0, 0), "y": (0, 0)}


def test_ensemble_of_unsplit_lengths(gpu):
    import torch
    cf = gpu
    probs = [_problem(cf, (Nx, 9, 6)) for Nx in (216, 44, 32)]
    states = [cf.perturbation_state(p, 0.05, seed=i) for i, p in enumerate(probs)]
    own = [s.copy() for s in states]
    for p, s in zip(probs, own):
        cf.step_(p.scheme, p.nlterm, s.velocity, s.stagepressure, 0.0, nsteps=3, **p.constraint)
    for tune in (False, True):
        runs = [s.copy() for s in states]
        cf.Ensemble(probs, runs, tune=tune).advance(3)
        torch.cuda.synchronize()
        for a, b in zip(runs, own):
            assert torch.equal(a.velocity, b.velocity) and torch.equal(a.stagepressure, b.stagepressure), tune
