"""Near lists (k_legs) made at positions that are not those of the build: a
program that builds the lists and then steps (fib_step moves the atoms before
its first force evaluation) must not lose a pair that the first step took
apart and the next steps bring back.

Pairs i, j beyond the cutoff fly apart by 0.9 delta in the first step, bounce
off a pinned atom each, and come together by 0.9 delta of their distance at
the build: within the cutoff, while no atom was ever farther than delta / 2
from its place at the build (45 such systems of several distances, far apart
in one box).  Forces after every step against those of a new handle at the
same positions, which sums the same terms: 1e-12 of the largest in FP64, 1e-6
in the mixed mode."""
import numpy as np
import pytest

from fib_md_amd import configs

pytestmark = pytest.mark.gpu

SIGMA, A, LISTFAC, TS = 2.0951e-10, 1.8, 2.0, 2e-14
CUT = 0.999 * A * SIGMA
GATE = 1.001 * CUT * 1.0005  # (the pair pass's range, rounded up)
DELTA = 0.1 * (LISTFAC * A * SIGMA - CUT)


def _systems():
    """k1, i, j, k2 along x in every system; k1 and k2 pinned."""
    L = (100e-10, 120e-10, 600e-10)
    d0 = GATE + 0.13 * DELTA
    X, V = [], []
    for s in range(45):
        y, z = (20 + 20 * (s % 5)) * 1e-10, (15 + 20 * (s // 5)) * 1e-10
        b = (2.335 + 0.05 * s / 44) * 1e-10  # i - k1 and j - k2
        v = 0.45 * DELTA / TS
        mid = 0.5 * L[0]
        for x, u in ((mid - 0.5 * d0 - b, 0.0), (mid - 0.5 * d0, -v), (mid + 0.5 * d0, v),
                     (mid + 0.5 * d0 + b, 0.0)):
            X.append((x, y, z))
            V.append((u, 0.0, 0.0))
    X, V = np.asfortranarray(X), np.asfortranarray(V)
    xs = np.tile([1, 0, 0, 1], 45).astype(np.int32)
    return X, V, xs, L


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lists_made_after_a_step_miss_no_pair(precision):
    from fib_md_amd import FibGPU
    from fib_md_amd.gpu import default_params, run_params_from_siga
    X, V, xs, L = _systems()
    n = len(X)
    at = np.ones(n, np.int32)
    p = default_params()
    p.listfac = LISTFAC
    run = dict(ts_i=TS, ts_r=TS, ttar1=300.0, ke_limit_1=600.0, tau_i=1e-13, tau_r=1e-13, teps=30.0,
               ntlist_i=1000, ntlist_r=1000, atlist_i=1000, atlist_r=1000, dslist_i=1000, dslist_r=1000,
               atm_out_i=1000, atm_out_r=1000, res_out=-5000, outz=(1.3, 3.5, 7.5, 9.8),
               atomz=(4.5, 6.5), ionz=5.5, sidewidth=0.1, dti=1e-9)
    g = FibGPU([(n, n, 0, L)], precision=precision, params=p)
    for again in range(2):  # the second time with forces of zero and no evaluation before the step
        g.set_state(X, V=V, atype=at, xsides=xs, Xi=X)
        g.build_nlist()
        if again == 0:
            g.set_run(run_params_from_siga(run))
            g.tint_init()
            g.ti_begin(2)
    near = np.ones(45, bool)  # systems whose i and j stayed within delta / 2
    out1 = hit = None
    tol = 1e-12 if precision == "fp64" else 1e-6
    for step in range(1, 5):
        assert g.step(2, max_steps=1).steps_done == 1
        Xg, _, F = g.state()
        d = np.linalg.norm(Xg - X, axis=1).reshape(45, 4)[:, 1:3].max(1)
        near &= d < 0.499 * DELTA
        r = np.linalg.norm((Xg[2::4] - Xg[1::4]), axis=1)
        if step == 1:
            out1 = r > GATE + 1.01 * DELTA
        hit = near & out1 & (r < CUT - 0.25 * DELTA)
        ref = FibGPU([(n, n, 0, L)], precision=precision, params=p)
        ref.set_state(Xg, atype=at, xsides=xs, Xi=X)
        ref.build_nlist()
        Fr = ref.force()["F"]
        ref.close()
        err = np.abs(F - Fr).max() / np.abs(Fr).max()
        print(f"{precision} step {step}: {int(hit.sum())} pairs came back, error {err:.2e}", flush=True)
        if step == 3:
            assert hit.sum() >= 5
        assert err <= tol
    g.close()
