"""The vertex pass with 64 atoms per wavefront (large batches, and other tiles
than the default) where a wavefront has more legs than its owner table holds,
so that it takes them in several runs, and several write-outs: second
neighbours in range (about 16 legs an atom, 1,000 a wavefront), with vacancies
(none to a dozen), with and without Ge.

The same periodic system in the small split and in the wide one: bit for bit
where the tiles choose it, and copies of it side by side (100,000 atoms and
more) against the oracle of one, FP64 at 1e-10 of max |F|, the mixed mode at 1e-6 of
the norm (as the vertex pass of small batches is)."""
import numpy as np
import pytest

from tests import gpu_common as gc

pytestmark = pytest.mark.gpu

SIGMA = 2.0951e-10
COPIES = {"many": (5, 5, 4), "vacancies": (5, 6, 4)}


def _box(kind, ge):
    from fib_md_amd import configs
    rng = np.random.default_rng(78)
    a, noise, keep = (5.15e-10, 0.05e-10, 1.0) if kind == "many" else (5.25e-10, 0.15e-10, 0.75)
    n = 5 if kind == "many" else 6
    X = configs.diamond(n, n, n, a)
    X = X[rng.random(len(X)) < keep]
    X = np.mod(X + rng.normal(0.0, noise, X.shape), n * a)
    at = np.ones(len(X), np.int32)
    return X, gc.with_ge(at, 0.3, 4) if ge else at, (n * a,) * 3


def _legs(X, L):
    d = X[:, None, :] - X[None, :, :]
    d -= np.round(d / L[0]) * L[0]
    r = np.sqrt((d * d).sum(2))
    return ((r < 0.999 * 1.8 * SIGMA) & (r > 0)).sum(1)


@pytest.mark.parametrize("ge", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["many", "vacancies"])
def test_tiles_give_the_same_bits(kind, precision, ge):
    X, at, L = _box(kind, ge)
    g = gc.gpu_system(X, at, L, len(X), 0, precision=precision)
    small = g.force()["F"]
    if kind == "many":
        assert _legs(X, L).mean() * 64 > 2 * 384
    for tiles in ((128, 4, 0), (128, 2, 0), (256, 2, 0)):
        print(kind, precision, ge, tiles, flush=True)
        g.set_tiles(*tiles)
        g.build_nlist()  # (the slots that the first pass keeps are worked out again)
        for _ in range(2):
            np.testing.assert_array_equal(g.force()["F"], small)
    g.close()


@pytest.mark.parametrize("ge", [False, True])
@pytest.mark.parametrize("kind", ["many", "vacancies"])
def test_copies_against_the_oracle_of_one(oracle_lib, kind, ge):
    X, at, L = _box(kind, ge)
    grid = COPIES[kind]
    n, m = len(X), int(np.prod(grid))
    shift = np.stack(np.meshgrid(*[np.arange(c) for c in grid], indexing="ij"), -1).reshape(-1, 3)
    assert n * m > 98304
    Xa = (X[None] + (shift * np.array(L))[:, None]).reshape(-1, 3)
    La = tuple(c * l for c, l in zip(grid, L))
    o = gc.oracle_system(X, at, L, n, 0)
    Fo, Wo = o.si_force(X, virial=True)
    Uo, _ = o.si_potential(X)
    fmax, wmax = np.abs(Fo).max(), np.abs(Wo).max()
    for precision in ("fp64", "mixed"):
        tu, tw = (1e-12, 1e-10) if precision == "fp64" else (1e-6, 1e-5)
        g = gc.gpu_system(Xa, np.tile(at, m), La, n * m, 0, precision=precision)
        plain = g.force()["F"]
        for en, vir in ((True, False), (False, True), (True, True)):
            print(kind, precision, ge, en, vir, flush=True)
            r = g.force(energy=en, virial=vir)
            np.testing.assert_array_equal(r["F"], plain)
            if en:
                assert abs(r["utot"] - m * Uo) <= tu * abs(m * Uo)
            if vir:
                assert np.abs(r["virial"] - m * Wo).max() <= tw * m * wmax
        F = plain.reshape(m, n, 3)
        if precision == "fp64":
            assert np.abs(F - Fo).max() <= 1e-10 * fmax
        else:
            assert np.linalg.norm(F - Fo) <= 1e-6 * np.linalg.norm(Fo) * np.sqrt(m)
        g.close()
