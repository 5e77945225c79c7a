"""Batches of trajectories (nbg_batch_cartesian) on the launches that give a
system two or three waves, few systems and more than compute units, body
counts mixed and runs of unequal length down to one step: with and without the
Jacobian, its records in both row updates, and a batch whose small class holds
a system that stays on one wave.  The reference row update gives the oracle's
bits; the factored one re-associates sums, whose results may differ by the
1e-10 of an array's largest entry that test_gpu_row_update.py asks for (x and v
read neither, their bits are the oracle's)."""
import numpy as np
import pytest

import oracle_lib as O
import nbodygradient_amd as nb
from nbodygradient_amd import workloads as W
from nbodygradient_amd.batch import cartesian_batch

pytestmark = pytest.mark.gpu

STATE = ("t", "x", "v", "xerror", "verror")
JAC = ("jac_step", "jac_error")


def _specs(ns, seed):
    rng = np.random.default_rng(seed)
    return [W.c2_system(rng, n) for n in ns]


@pytest.mark.parametrize("copies", [1, 45])  # 7 systems; 315, more than compute units
@pytest.mark.parametrize("form", ["reference", "factored", "no gradient", "one kicked"])
def test_batched_trajectories(form, copies):
    print("gpu: batched trajectories, %s, %d copies" % (form, copies), flush=True)
    ns, N = [3, 6, 7, 8, 10, 11, 12], [4, 1, 6, 3, 2, 5, 3]
    specs = _specs(ns, 700)
    states = W.initial_states(specs, processes=1)
    pair = [np.zeros((n, n), dtype=np.uint8, order="F") for n in ns]
    if form == "one kicked":
        pair[1][2, 4] = pair[1][4, 2] = 1
    jac = form != "no gradient"
    ctx = nb.default_context()
    ctx.set_row_update(1 if form == "factored" else 0)
    try:
        got = cartesian_batch(specs * copies, N * copies, states=states * copies, grad=jac, jacobian=jac,
                              pair=pair * copies if form == "one kicked" else None)
    finally:
        ctx.set_row_update(0)
    assert len(got) == copies * len(ns)
    for q, s in enumerate(specs):
        x, v, j = states[q]
        os_ = O.OState(x, v, s.elements[:, 0], t=s.t0, jac_init=j, pair=pair[q])
        rec = O.cartesian_output(os_, s.h, s.tmax, N[q])
        for r in (got[q], got[q + (copies - 1) * len(ns)]):
            for key in STATE:
                assert np.array_equal(r[key], rec[key]), (s.n, key)
            for key in JAC if jac else ():
                if form != "factored":
                    assert np.array_equal(r[key], rec[key]), (s.n, key)
            if form == "factored":
                big = np.max(np.abs(rec["jac_step"]))
                assert np.max(np.abs(r["jac_step"] - rec["jac_step"])) <= 1e-10 * big
                assert np.max(np.abs(r["jac_error"])) <= 1e-15 * big
