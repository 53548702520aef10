"""Two atoms at one place show in the results, alone and among others: an
infinite energy of each and in total (the repulsion of the pair, B / r^4),
and no finite force on them.  Atoms out of their range are as without them:
the same bits, alone and in a box with the pair."""
import numpy as np
import pytest

from fib_md_amd import configs

pytestmark = pytest.mark.gpu


def _evaluate(X, L, precision, at):
    from fib_md_amd import FibGPU
    g = FibGPU([(len(X), len(X), 0, L)], precision=precision)
    g.set_state(X, atype=at)
    g.build_nlist()
    plain = g.force()["F"]
    r = g.force(energy=True, virial=True)
    g.close()
    np.testing.assert_array_equal(plain, r["F"])
    return r


@pytest.mark.parametrize("ge", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_isolated_pair(precision, ge):
    L = (60e-10, 50e-10, 40e-10)
    far = np.array([[30e-10, 30e-10, 30e-10], [32.4e-10, 30e-10, 30e-10]])
    X = np.vstack([far, [[7e-10, 8e-10, 9e-10]] * 2])
    at = np.array([1, 1, 1, 2 if ge else 1], np.int32)
    r = _evaluate(X, L, precision, at)
    own = _evaluate(far, L, precision, at[:2])
    print(precision, r["F"], r["u"], r["utot"], flush=True)
    assert np.isnan(r["F"][2:]).all()
    assert np.isposinf(r["u"][2:]).all() and np.isposinf(r["utot"])
    np.testing.assert_array_equal(r["F"][:2], own["F"])
    np.testing.assert_array_equal(r["u"][:2], own["u"])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_pair_in_a_crystal(precision):
    n = 4
    L = (n * configs.A_SI,) * 3
    X = configs.perturbed_crystal(n, 0.05e-10, 3)
    X = np.vstack([X, X[100]])
    r = _evaluate(X, L, precision, np.ones(len(X), np.int32))
    print(precision, r["F"][[100, -1]], r["u"][[100, -1]], r["utot"], flush=True)
    assert not np.isfinite(r["F"][[100, -1]]).any()
    assert not np.isfinite(r["u"][[100, -1]]).any() and not np.isfinite(r["utot"])
    d = X - X[100]
    d -= np.round(d / L[0]) * L[0]
    out = np.linalg.norm(d, axis=1) > 2 * 1.8 * 2.0951e-10  # no term with one of the two
    assert out.sum() > 100 and np.isfinite(r["F"][out]).all() and np.isfinite(r["u"][out]).all()
