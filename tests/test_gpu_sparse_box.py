"""List builds in boxes of many more cells than atoms (clusters in vacuum):
runs of empty cells, and scans over buckets of which most hold nothing.  The
lists against all pairs within the list radius, for builds that follow each
other as the atoms move, and energies and forces the same bits as in a batch
with a dense crystal."""
import numpy as np
import pytest

from fib_md_amd import configs

pytestmark = pytest.mark.gpu

RC = 1.1 * 1.8 * 2.0951e-10


def _clusters(L, n, seed):
    """n clusters of a few atoms, some across the faces of the box."""
    rng = np.random.default_rng(seed)
    at0 = configs.diamond(2, 1, 1)
    c = rng.random((n, 3)) * np.array(L)
    c[: n // 4, 0] = 0.0
    c[n // 4: n // 2, 1] = L[1] - 1e-10
    X = (c[:, None] + at0[None] + rng.normal(0.0, 0.05e-10, (n, len(at0), 3))).reshape(-1, 3)
    return np.mod(X, np.array(L))


def _pairs(X, L):
    from scipy.spatial import cKDTree
    p = cKDTree(X, boxsize=L).query_pairs(RC, output_type="ndarray")
    return {(min(a, b), max(a, b)) for a, b in p.tolist()}


def _listed(g):
    s2, _ = g.half_sets()
    return {(i, j - 1) for i, js in enumerate(s2) for j in js}


# cells: 3 x 3 x 20,000; 241 x 241 x 48 (2.8 million); 100 x 3 x 3; two atoms'
# worth of buckets past a multiple of the scan's chunks; boxes of two cells a side; 17.2
# million, more than 8,192 chunks
@pytest.mark.parametrize("cells,n", [((3, 3, 20000), 40), ((241, 241, 48), 60), ((100, 3, 3), 30),
                                     ((32, 16, 16), 20), ((2, 2, 5000), 30), ((2, 600, 600), 40),
                                     ((262, 257, 256), 60)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lists_of_clusters_in_vacuum(cells, n, precision):
    pytest.importorskip("scipy")
    from fib_md_amd import FibGPU
    L = tuple((c + 0.5) * RC for c in cells)
    X = _clusters(L, n, 21)
    at = np.ones(len(X), np.int32)
    g = FibGPU([(len(X), len(X), 0, L)], precision=precision)
    assert tuple(g.cells()) == cells
    rng = np.random.default_rng(3)
    for _ in range(3):
        g.set_state(X, atype=at)
        g.build_nlist()
        want, have = _pairs(X, L), _listed(g)
        if min(cells) > 2:
            assert have == want
        else:
            assert have <= want
        r = g.force(energy=True)
        assert np.isfinite(r["F"]).all() and np.isfinite(r["utot"])
        X = np.mod(X + rng.normal(0.0, 0.02e-10, X.shape), np.array(L))
    # the same beside a crystal
    C = configs.perturbed_crystal(4, 0.05e-10, 5)
    LC = (4 * configs.A_SI,) * 3
    b = FibGPU([(len(C), len(C), 0, LC), (len(X), len(X), 0, L), (len(C), len(C), 0, LC)],
               precision=precision)
    for k, (Y, a) in enumerate(((C, np.ones(len(C), np.int32)), (X, at), (C, np.ones(len(C), np.int32)))):
        b.set_state(Y, atype=a, inst=k)
    g.set_state(X, atype=at)
    g.build_nlist()
    b.build_nlist()
    g.compute(energy=True)
    b.compute(energy=True)
    alone, other = g.forces(0, energy=True), b.forces(1, energy=True)
    np.testing.assert_array_equal(alone["F"], other["F"])
    np.testing.assert_array_equal(alone["u"], other["u"])
    assert alone["utot"] == other["utot"] and b.forces(0)["utot"] == b.forces(2)["utot"]
    g.close()
    b.close()
