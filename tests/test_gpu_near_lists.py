"""Near lists of the pair pass (k_legs): between list builds the pass runs
over the row entries that were within cutoff + delta at the build, except
around atoms that moved more than delta / 2.  Forces of the MD steps are
compared with those of a new handle at the same positions, whose first pass
after its build reads the whole rows: in a cold slab with a fast recoil (near
lists everywhere but in its cascade), a hot one (every atom leaves its near
list between builds) and a compressed one (more near entries than a near
list holds), two instances in a batch that rebuild at different steps.

A pair left out of either would change its atoms' forces by far more than
rounding.  Both sides sum the same terms in another order: FP64 within 1e-12
of the forces' norm; mixed within 1e-6 (the FP32 terms' rounding, 2e-7 of
their size each, where the sums cancel)."""
import numpy as np
import pytest

from fib_md_amd import configs

pytestmark = pytest.mark.gpu


def _slab(kind, seed):
    a = 5.1e-10 if kind == "dense" else configs.A_SI
    s = configs.si_slab(6, seed, nz=5, T=4000.0 if kind == "hot" else 300.0, a=a)
    rng = np.random.default_rng(seed + 5)
    free = (s["xsides"] == 0) & (s["atype"] < 3)
    s["X0"] = s["X"].copy()
    s["X"] = np.mod(s["X"] + np.where(free[:, None], rng.normal(0.0, 0.05e-10, s["X"].shape), 0.0),
                    np.array(s["L"]))
    return s


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["cold", "hot", "dense"])
def test_near_lists_miss_no_pair(kind, prec):
    from fib_md_amd import FibGPU
    slabs = [_slab(kind, 31), _slab(kind, 32)]
    desc = [(len(s["X"]), s["nsg"], s["nlj"], s["L"]) for s in slabs]
    # a recoil (200 eV Si) in the first instance only: it rebuilds more often
    slabs[0]["V"][700] = [2.2e4, 1.1e4, -2.8e4]
    g = FibGPU(desc, precision=prec)
    for k, s in enumerate(slabs):
        g.set_state(s["X"], V=s["V"], atype=s["atype"], xsides=s["xsides"], Xi=s["X0"], inst=k)
    g.md_begin([s["surface_z"] for s in slabs], [s["bottom_z"] for s in slabs])
    tol = 1e-12 if prec == "fp64" else 1e-6
    for chunk in (1, 2, 3, 5, 11, 23):
        g.md_run(chunk)
        ref = FibGPU(desc, precision=prec)
        st = [g.state(k) for k in range(2)]
        for k, s in enumerate(slabs):
            ref.set_state(st[k][0], atype=s["atype"], inst=k)
        ref.build_nlist()
        ref.compute()
        for k in range(2):
            F, Fr = st[k][2], ref.forces(k)["F"]
            d = np.linalg.norm(F - Fr) / np.linalg.norm(Fr)
            print(f"{kind} {prec} +{chunk} steps, instance {k}: {d:.2e}, "
                  f"builds {g.md_report(k)['builds']}", flush=True)
            assert d <= tol
        ref.close()
    b = [g.md_report(k)["builds"] for k in range(2)]
    g.close()
    assert b[0] > b[1] or kind == "hot"
