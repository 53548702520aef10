"""Energies and virial of every instance of a batch that holds an instance of
more than 524,288 atoms (reduced in several chunks, a workgroup each) beside
small ones (one chunk, and no work for those workgroups): the same as each
instance gives alone.

The order of the sums differs with the batch at most: 1e-12 of the energy
(4.5e6 terms, sqrt(4.5e6) 2^-53 = 2e-13), 1e-11 of the virial, whose terms
cancel to a hundredth of their sizes."""
import numpy as np
import pytest

from fib_md_amd import configs

pytestmark = pytest.mark.gpu


def _crystal(n, seed):
    rng = np.random.default_rng(seed)
    L = tuple(configs.A_SI * c for c in n)
    X = configs.diamond(*n)
    X = np.mod(X + rng.normal(0.0, 0.05e-10, X.shape), L)
    # a Ga at a hexagonal interstitial site
    X = np.vstack([X, [[1.625 * configs.A_SI] * 3]])
    at = np.concatenate([np.ones(len(X) - 1, np.int32), [3]]).astype(np.int32)
    return X, at, L


def _evaluate(systems, precision):
    from fib_md_amd import FibGPU
    g = FibGPU([(len(X), len(X) - 1, 1, L) for X, _, L in systems], precision=precision)
    for k, (X, at, _) in enumerate(systems):
        g.set_state(X, atype=at, Xi=X, inst=k)
        g.set_impact(1, inst=k)
    g.build_nlist()
    g.compute(energy=True, virial=True)
    out = [g.forces(k, energy=True, virial=True) for k in range(len(systems))]
    g.md_begin([s[2][2] for s in systems], [0.0] * len(systems))
    epot = g.md_energy()
    g.close()
    return out, epot


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_small_instances_beside_one_of_several_chunks(precision):
    systems = [_crystal((4, 4, 4), 1), _crystal((41, 40, 40), 2), _crystal((6, 5, 4), 3),
               _crystal((3, 3, 3), 4)]
    assert len(systems[1][0]) > 524288 and all(len(s[0]) < 65536 for s in systems[2:])
    out, epot = _evaluate(systems, precision)
    for k, s in enumerate(systems):
        (own,), (e,) = _evaluate([s], precision)
        print(f"{precision} instance {k}, {len(s[0])} atoms: utot {out[k]['utot']!r} "
              f"alone {own['utot']!r}", flush=True)
        np.testing.assert_array_equal(out[k]["F"], own["F"])
        np.testing.assert_array_equal(out[k]["u"], own["u"])
        assert abs(out[k]["utot"] - own["utot"]) <= 1e-12 * abs(own["utot"])
        assert abs(epot[k] - e) <= 1e-12 * abs(e)
        assert np.abs(out[k]["virial"] - own["virial"]).max() <= 1e-11 * np.abs(own["virial"]).max()


# beside a 4 x 4 x 4 crystal (513 atoms): a batch of up to 98,304 atoms, one
# of more (another split of the vertex pass), and instances just below and
# above that size themselves
@pytest.mark.parametrize("other", [(9, 8, 7), (24, 23, 22), (32, 24, 16), (25, 25, 26), (5, 5, 41)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_energies_and_virial_have_the_bits_of_the_instance_alone(other, precision):
    """Sums within an instance have an order that depends on it alone."""
    systems = [_crystal((4, 4, 4), 11), _crystal(other, 12), _crystal((26, 26, 25), 13)]
    for batch in (systems[:2], systems):
        out, epot = _evaluate(batch, precision)
        for k, s in enumerate(batch):
            (own,), (e,) = _evaluate([s], precision)
            print(f"{precision} {len(s[0])} atoms: {out[k]['utot']!r} {own['utot']!r}", flush=True)
            assert out[k]["utot"] == own["utot"] and epot[k] == e
            np.testing.assert_array_equal(out[k]["u"], own["u"])
            np.testing.assert_array_equal(out[k]["virial"], own["virial"])
