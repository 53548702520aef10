"""An instance gives the same bits alone and in any batch, whatever sort and
whatever reductions the batch takes: one workgroup per instance sorts up to
8,192 atoms and cells (k_sort_small), the scans and scatters sort more; up to
eight instances of at most 65,536 atoms are reduced where the next kernel
decides, more of them by a launch of their own, larger ones in chunks; small
batches have eight or 16 atoms per wavefront in the vertex pass, large ones 64."""
import numpy as np
import pytest

from fib_md_amd import configs
from tests import gpu_common as gc

pytestmark = pytest.mark.gpu

SMALL = (4, 4, 4)
STEPS = 40


def _slab(n, seed):
    rng = np.random.default_rng(seed)
    X = configs.diamond(*n)
    L = tuple(configs.A_SI * c for c in n)
    X = np.mod(X + rng.normal(0.0, 0.05e-10, X.shape), L)
    V = rng.normal(0.0, 420.0, X.shape)
    X = np.vstack([X, [[1.625 * configs.A_SI] * 3]])
    V = np.vstack([V, np.zeros(3)])
    at = np.concatenate([np.ones(len(X) - 1, np.int32), [3]]).astype(np.int32)
    return X, V, at, L


def _run(slabs, precision):
    from fib_md_amd import FibGPU
    g = FibGPU([(len(X), len(X) - 1, 1, L) for X, _, _, L in slabs], precision=precision)
    for k, (X, V, at, L) in enumerate(slabs):
        g.set_state(X, V=V, atype=at, Xi=X, inst=k)
    g.md_begin([s[3][2] for s in slabs], [0.0] * len(slabs))
    for k, (_, _, _, L) in enumerate(slabs):
        g.md_fire(k, 1, np.array([0.5 * L[0], 0.4 * L[1], 0.55 * L[2]]),
                  np.array([0.0, 1.0e4, -5.0e4]))
    g.md_run(STEPS)
    out = []
    epot = g.md_energy()
    for k in range(len(slabs)):
        r = g.md_report(k)
        X, V = g.state(k)[:2]
        out.append((np.asarray(X), np.asarray(V), r, epot[k]))
    g.close()
    return out


# sizes beside the 4 x 4 x 4 slab under test (513 atoms)
BATCHES = {
    "eight": [SMALL] * 7,
    "nine": [SMALL] * 8,
    "sort_8185": [(3, 11, 31)],
    "sort_8192_and_ion": [(8, 8, 16)],
    "sort_8201": [(5, 5, 41)],
    "chunks": [(21, 20, 20)],
    "vertex_pass_of_64": [(26, 26, 26)],
}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_alone_and_in_a_batch(name, precision):
    own = _slab(SMALL, 5)
    rest = [_slab(n, 100 + k) for k, n in enumerate(BATCHES[name])]
    print(f"{name}: {[len(s[0]) for s in rest]} atoms", flush=True)
    alone = _run([own], precision)[0]
    batch = _run([own] + rest, precision)
    assert alone[2]["steps"] == STEPS
    np.testing.assert_array_equal(batch[0][0], alone[0])
    np.testing.assert_array_equal(batch[0][1], alone[1])
    assert batch[0][2] == alone[2]
    # (the vertex pass's workgroups, and with them the order of the sum of up
    # to 1.4e5 terms, depend on the batch: sqrt(1.4e5) 2^-53 = 4e-14 of it)
    assert abs(batch[0][3] - alone[3]) <= 1e-12 * abs(alone[3])
    if len(rest) == 1:  # and the other one
        other = _run(rest, precision)[0]
        np.testing.assert_array_equal(batch[1][0], other[0])
        np.testing.assert_array_equal(batch[1][1], other[1])
        assert batch[1][2] == other[2]
        assert abs(batch[1][3] - other[3]) <= 1e-12 * abs(other[3])


@pytest.mark.parametrize("n", [(3, 11, 31), (8, 8, 16), (5, 5, 41)])
def test_sort_sizes_against_the_oracle(oracle_lib, n):
    X, _, at, L = _slab(n, 9)
    m = len(X)
    o = gc.oracle_system(X, at, L, m - 1, 1, impact=1)
    Fo = o.si_force(X)
    ref2, reflj = o.half_sets()
    g = gc.gpu_system(X, at, L, m - 1, 1)
    F = g.force(impact=1)["F"]
    s2, slj = g.half_sets()
    g.close()
    assert s2 == ref2 and slj == reflj
    assert np.abs(F - Fo).max() <= 1e-10 * np.abs(Fo).max()
