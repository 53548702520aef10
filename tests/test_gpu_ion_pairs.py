"""Moliere pairs worked off by a whole wavefront (k_legs): one ion, ions that
share a cell (more pairs in a wavefront than it has lanes, Ga-Ga pairs), ions
of which some are not yet fired.

FP64 against the oracle at the parity tests' bounds (1e-10 of max |F| and of
max |W|, 1e-12 of U).  Mixed: the pairs beyond mixed_r64 are FP32, about ten
operations rounded at 2^-24 each, so 1e-6 of the norm of the forces.  The oracle's U is
the reference's si_potential, which counts ions not yet fired too
(si.f90:278-368; the forces leave them out): compared where all are fired."""
import numpy as np
import pytest

from fib_md_amd import configs
from tests import gpu_common as gc

pytestmark = pytest.mark.gpu


def _case(nions, seed):
    rng = np.random.default_rng(seed)
    a, n = configs.A_SI, 4
    L = (n * a,) * 3
    X = configs.diamond(n, n, n, a)
    X = np.mod(X + rng.normal(0.0, 0.1e-10, X.shape), n * a)
    ions = []
    while len(ions) < nions:  # all in one cell, 0.8 A from everything
        x = (1.1 + 0.9 * rng.random(3)) * a
        if min(np.linalg.norm(y - x) for y in list(X) + ions) > 0.8e-10:
            ions.append(x)
    at = np.concatenate([np.ones(len(X), np.int32), np.full(nions, 3, np.int32)])
    return np.vstack([X, ions]), at, L, len(X)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nions,impact", [(1, 1), (7, 7), (7, 3), (7, 0)])
def test_ion_pairs(oracle_lib, nions, impact, precision):
    X, at, L, nsg = _case(nions, 40 + nions)
    o = gc.oracle_system(X, at, L, nsg, nions, impact=impact)
    Fo, Wo = o.si_force(X, virial=True)
    Uo, _ = o.si_potential(X)
    g = gc.gpu_system(X, at, L, nsg, nions, precision=precision)
    lj = g.half_sets()[1]
    print(f"{nions} ions, {impact} fired: {len(lj)} listed ion pairs", flush=True)
    plain = g.force(impact)
    full = g.force(impact, energy=True, virial=True)
    g.close()
    if nions > 1:
        assert len(lj) > 2 * 64
    np.testing.assert_array_equal(plain["F"], full["F"])
    if precision == "fp64":
        assert np.abs(full["F"] - Fo).max() <= 1e-10 * np.abs(Fo).max()
        if impact == nions:
            assert abs(full["utot"] - Uo) <= 1e-12 * abs(Uo)
        assert np.abs(full["virial"] - Wo).max() <= 1e-10 * np.abs(Wo).max()
    else:
        assert np.linalg.norm(full["F"] - Fo) <= 1e-6 * np.linalg.norm(Fo)
        if impact == nions:
            assert abs(full["utot"] - Uo) <= 1e-6 * abs(Uo)
