"""Host transfers at the sizes where their path changes: one copy up to 2 MiB,
then chunks of 256 KiB to 2 MiB through up to four lanes; the arrays are given
back bit for bit, on a handle used for the first time, reused, and from two
threads with a handle each."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 400e-10


def _state(n, seed):
    rng = np.random.default_rng(seed)
    X = rng.random((n, 3)) * L
    return X, rng.normal(0.0, 500.0, (n, 3)), np.where(rng.random(n) < 0.3, 2, 1).astype(np.int32)


def _round_trip(g, n, seed, inst=0, with_v=True):
    X, V, at = _state(n, seed)
    g.set_state(X, V=V if with_v else None, atype=at, inst=inst,
                xsides=np.zeros(n, np.int32) if with_v else None, Xi=X if with_v else None)
    gX, gV, gF = g.state(inst)
    np.testing.assert_array_equal(gX, X)
    np.testing.assert_array_equal(gV, V if with_v else np.zeros_like(V))
    np.testing.assert_array_equal(gF, np.zeros_like(V))


# 29,127 and 29,130 atoms: 72 B each, either side of 2 MiB in state(); 26,214
# and 26,215: 80 B in set_state; 349,525 and 349,526: X of whole chunks and one
# more atom; 262,144: more chunks than lanes
@pytest.mark.parametrize("n", [1, 3277, 26214, 26215, 29127, 29130, 87382, 262144, 349525, 349526])
def test_round_trip(n):
    from fib_md_amd import FibGPU
    print(n, flush=True)
    g = FibGPU([(n, n, 0, (L, L, L)), (7, 7, 0, (L, L, L))], precision="mixed")
    for seed in (1, 2):
        _round_trip(g, n, seed, with_v=seed == 1)
        _round_trip(g, 7, seed, inst=1)
    # refused as before: a wrong species anywhere, and nothing is changed
    X, V, at = _state(n, 9)
    for k in {0, n // 2, n - 1}:
        for t in (0, 3, -1, 2**31 - 1):
            bad = at.copy()
            bad[k] = t
            with pytest.raises(Exception, match="atype"):
                g.set_state(X, V=V, atype=bad)
    np.testing.assert_array_equal(g.state()[0], _state(n, 2)[0])
    g.close()


def test_round_trip_from_two_threads():
    from fib_md_amd import FibGPU
    err = []

    def work(k):
        try:
            n = 150000 + k
            g = FibGPU([(n, n, 0, (L, L, L))], precision="fp64")
            for seed in range(4):
                _round_trip(g, n, 10 * k + seed)
            g.close()
        except BaseException as e:
            err.append(e)

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not err, err
