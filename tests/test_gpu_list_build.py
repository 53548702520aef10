"""The list build (k_nbuild) in every path of a cell: halos that fit two
candidates per lane with one or two registers of them left after the box
filter, denser ones, boxes of few cells (no unique periodic shift), cells at
the faces of larger ones (shifts of +-L), wide cells (three candidates per
lane, or more than are kept), positions outside the box, Ga ions
among the candidates, empty cells; and 1 to 16 cells per wavefront.

Neighbour sets equal the oracle's; FP64 forces agree with it within 1e-10 of
max |F| (the parity tests' bound), which also takes the stencil bookkeeping
through the vertex pass's partner lookups."""
import numpy as np
import pytest

from fib_md_amd import configs
from tests import gpu_common as gc

pytestmark = pytest.mark.gpu

# cells, lattice constant (A), noise (A), fraction kept, ions, box shifts
CASES = {
    "wide": ((19, 13, 4), 5.431, 0.12, 1.0, 4, False),
    "three_cells": ((3, 3, 3), 5.431, 0.1, 1.0, 2, False),
    "flat": ((14, 3, 4), 5.431, 0.1, 1.0, 0, False),
    "dense": ((6, 6, 6), 4.95, 0.05, 1.0, 3, False),
    "very_dense": ((7, 6, 6), 4.5, 0.02, 1.0, 2, False),
    "wide_cells": ((7, 6, 6), 5.431, 0.1, 1.0, 3, False),
    "wide_cells_outside": ((6, 5, 7), 5.431, 0.05, 1.0, 2, True),
    "wide_cells_dense": ((6, 6, 6), 5.1, 0.02, 1.0, 0, False),
    "sparse": ((8, 8, 8), 5.431, 0.2, 0.25, 6, False),
    "outside_the_box": ((18, 5, 5), 5.431, 0.1, 1.0, 3, True),
}


def _system(name):
    n, a, noise, keep, nions, shifted = CASES[name]
    a, noise = a * 1e-10, noise * 1e-10
    rng = np.random.default_rng(sum(map(ord, name)))
    L = np.array(n) * a
    X = configs.diamond(*n, a=a)
    X = X[rng.random(len(X)) < keep]
    X = np.mod(X + rng.normal(0.0, noise, X.shape), L)
    nsg = len(X)
    cell = rng.choice(n[0] * n[1] * n[2], nions, replace=False)
    c = np.stack(np.unravel_index(cell, n), axis=1)
    X = np.vstack([X, np.mod((c + 0.625) * a, L)])
    if shifted:  # some atoms a box or two away (the reference takes them)
        k = rng.integers(-1, 3, X.shape) * (rng.random((len(X), 1)) < 0.1)
        X = X + k * L
    at = np.concatenate([np.ones(nsg, np.int32), np.full(nions, 3, np.int32)])
    return X, at, tuple(L), nsg, nions


@pytest.mark.parametrize("name", list(CASES))
def test_list_build_paths(oracle_lib, name):
    X, at, L, nsg, nlj = _system(name)
    print(f"{name}: {len(X)} atoms", flush=True)
    o = gc.oracle_system(X, at, L, nsg, nlj, impact=nlj)
    ref2, reflj = o.half_sets()
    Fo = o.si_force(X)
    from fib_md_amd import FibGPU
    g = FibGPU([(len(X), nsg, nlj, L)], precision="fp64")
    g.set_state(X, atype=at)
    for cells in (0, 4, 16):
        g.set_tiles(0, 0, cells)
        g.build_nlist()
        s2, slj = g.half_sets()
        assert s2 == ref2 and slj == reflj
        F = g.force(impact=nlj)["F"]
        assert np.abs(F - Fo).max() <= 1e-10 * np.abs(Fo).max()
    g.close()
