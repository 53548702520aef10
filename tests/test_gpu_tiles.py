"""Launch tiles: what a handle reports is what its launches take, whatever it
reports can be set, and the tuner tries the default of the handle's size."""
import numpy as np
import pytest

from fib_md_amd import configs

pytestmark = pytest.mark.gpu


def _handle(n, precision="mixed"):
    from fib_md_amd import FibGPU
    L = tuple(configs.A_SI * c for c in n)
    m = 8 * n[0] * n[1] * n[2]
    return FibGPU([(m, m, 0, L)], precision=precision)


# cells of the list build at 1.1 cutoffs: 1.309 per lattice constant
@pytest.mark.parametrize("n,cells", [((4, 4, 4), 1), ((24, 25, 24), 1), ((25, 25, 26), 2),
                                     ((40, 40, 40), 4), ((50, 50, 50), 8)])
def test_reported_tiles_can_be_set(n, cells):
    g = _handle(n)
    total = int(np.prod(g.cells()))
    assert cells == (1 if total < 32768 else 2 if total < 131072 else 4 if total < 262144 else 8)
    assert g.tiles() == (256, 4, cells)
    for nb in (1, 2, 4, 8, 16):
        g.set_tiles(0, 0, nb)
        assert g.tiles() == (256, 4, nb)
    g.set_tiles(0, 0, 0)
    own = g.tiles()
    g.set_tiles(*own)
    assert g.tiles() == own
    from fib_md_amd.gpu import GPUError
    for bad in ((64, 4, 8), (256, 3, 8), (256, 4, 3), (256, 4, 32), (256, 4, -1)):
        with pytest.raises(GPUError, match="tri_ns"):
            g.set_tiles(*bad)
    assert g.tiles() == own
    g.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tuner_tries_the_default(precision):
    from fib_md_amd import FibGPU, autotune
    n = (5, 5, 4)
    L = tuple(configs.A_SI * c for c in n)
    rng = np.random.default_rng(8)
    X = configs.diamond(*n)
    X = np.mod(X + rng.normal(0.0, 0.05e-10, X.shape), L)
    V = rng.normal(0.0, 420.0, X.shape)
    at = np.ones(len(X), np.int32)
    out = []
    for nb in (0, 1, 2, 8):
        g = FibGPU([(len(X), len(X), 0, L)], precision=precision)
        g.set_tiles(0, 0, nb)
        g.set_state(X, V=V, atype=at, Xi=X)
        g.md_begin([L[2]], [0.0])
        g.md_run(60)
        out.append(g.state())
        if nb == 8:
            best, table = autotune.tune_tiles(g, steps=4, warmup=1)
            tiles = [t for t, _ in table]
            assert (256, 4, 1) in tiles and best in tiles and g.tiles() == best
            g.set_tiles(*best)
        g.close()
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)
