"""The later rungs' queue of the persistent implicit solve, on cells that the
first rung does not solve: fewer cells than waves (one lane each, the rungs of
a cell side by side), a little over a wave's share, and enough for 64 lanes a
wave.  Outcome, rung, iterations and state of every cell equal the oracle's."""
import numpy as np
import pytest

import kzo
from koral_zig_amd import abi_types as T
from koral_zig_amd import hip, workloads

pytestmark = pytest.mark.gpu
FIELDS = ("ok", "rung", "iters", "whichprim", "whicheq", "whichframe")


@pytest.fixture(scope="module")
def hard():
    """(inputs, oracle results) of the cells of 20 000 that need a later rung
    or fail the whole ladder."""
    phys = T.physics_puffy()
    pp, geom, dt = workloads.implicit_batch_inputs(
        20000, 29, phys, lambda p, g: kzo.opac_entry(p, g, phys.gam, phys.opac)[:, 3])
    res, p, u = kzo.solve_implicit(pp, geom, dt, phys.gam, phys.rad, phys.opac, phys.implicit)
    pick = np.nonzero((res["rung"] != 0) | (res["ok"] == 0))[0]
    assert pick.size > 1500 and (res["ok"][pick] == 0).any() and (res["rung"][pick] == 2).any()
    return phys, pp[pick], geom[pick], dt[pick], res[pick], p[pick], u[pick]


@pytest.mark.parametrize("n", [1, 65, 1025, 40000])
def test_ladder_queue(hard, n):
    phys, pp, geom, dt, res, p, u = hard
    at = np.arange(n) % len(pp)
    b = hip.ImplicitBatch(n, phys)
    b.set(pp[at], geom[at], dt[at])
    print(f"{n} cells past the first rung", flush=True)
    for again in range(2):  # the second solve starts from what the first left in the work arrays
        b.solve()
        uu, po, r, (nfail, iters, solves) = b.get()
        for k in FIELDS:
            assert np.array_equal(r[k], res[k][at]), (again, k)
        ok = r["ok"] == 1
        assert po[ok].tobytes() == p[at][ok].tobytes() and uu[ok].tobytes() == u[at][ok].tobytes(), again
        assert np.array_equal(po[~ok], pp[at][~ok]), again
        assert (nfail, iters, solves) == (int((~ok).sum()), int(r["iters"][ok].sum()), int(ok.sum()))
    b.close()
