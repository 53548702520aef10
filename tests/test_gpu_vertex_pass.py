"""The vertex pass (k_tri) where its layout can go wrong: atoms with few legs
(cos + 1/3 shared between a pair's two legs), with more than the shared rows
hold (formed per term), both in one wavefront, atoms without any leg, and
more legs in a wavefront than its owner table holds; with and without Ge.

FP64 against the oracle at the parity tests' bounds (1e-10 of max |F|).  The
mixed mode against the oracle: a term's FP32 part is about ten operations on
values rounded once, so an atom's terms carry about sqrt(10) 2^-24 = 2e-7 of
their own size each, in random directions; 1e-6 of the norm of all forces
leaves room for terms a few times larger than the net forces."""
import numpy as np
import pytest

from fib_md_amd import configs
from tests import gpu_common as gc

pytestmark = pytest.mark.gpu

SIGMA = 2.0951e-10


def _case(name):
    rng = np.random.default_rng(77)
    if name == "few":  # four or five legs
        a, n, noise, keep = configs.A_SI, 5, 0.03e-10, 1.0
    elif name == "many":  # second neighbours in range: about 16 legs each
        a, n, noise, keep = 5.15e-10, 5, 0.05e-10, 1.0
    elif name == "both":  # vacancies and noise: none to a dozen legs
        a, n, noise, keep = 5.25e-10, 5, 0.15e-10, 0.6
    else:  # a thin gas of fragments: atoms without legs
        a, n, noise, keep = configs.A_SI, 6, 0.15e-10, 0.12
    X = configs.diamond(n, n, n, a)
    X = X[rng.random(len(X)) < keep]
    X = np.mod(X + rng.normal(0.0, noise, X.shape), n * a)
    return X, np.ones(len(X), np.int32), (n * a,) * 3


def _legs(X, L):
    d = X[:, None, :] - X[None, :, :]
    d -= np.round(d / L[0]) * L[0]
    r = np.sqrt((d * d).sum(2))
    return ((r < 0.999 * 1.8 * SIGMA) & (r > 0)).sum(1)


@pytest.mark.parametrize("ge", [0.0, 0.3])
@pytest.mark.parametrize("name", ["few", "many", "both", "gas"])
def test_vertex_pass(oracle_lib, name, ge):
    X, at, L = _case(name)
    if ge:
        at = gc.with_ge(at, ge, 3)
    n = len(X)
    legs = _legs(X, L)
    print(f"{name}: {n} atoms, legs {legs.min()} to {legs.max()}", flush=True)
    if name == "few":
        assert legs.max() <= 8
    if name == "many":
        assert legs.min() > 8 and legs.mean() * 64 > 384
    if name == "both":
        assert legs.min() <= 2 and legs.max() > 8
    if name == "gas":
        assert legs.min() == 0
    o = gc.oracle_system(X, at, L, n, 0)
    Fo, Wo = o.si_force(X, virial=True)
    Uo, _ = o.si_potential(X)
    fmax = np.abs(Fo).max()
    for prec in ("fp64", "mixed"):
        g = gc.gpu_system(X, at, L, n, 0, precision=prec)
        plain = g.force(0)  # the variant of the time steps
        full = g.force(0, energy=True, virial=True)
        g.close()
        np.testing.assert_array_equal(plain["F"], full["F"])
        if prec == "fp64":
            assert np.abs(full["F"] - Fo).max() <= 1e-10 * fmax
            assert abs(full["utot"] - Uo) <= 1e-12 * abs(Uo)
            assert np.abs(full["virial"] - Wo).max() <= 1e-10 * np.abs(Wo).max()
        else:
            assert np.linalg.norm(full["F"] - Fo) <= 1e-6 * np.linalg.norm(Fo)
            assert abs(full["utot"] - Uo) <= 1e-6 * abs(Uo)
