"""The one-wave launches (nbg_run, nbg_run_duo) against the oracle.  A class of
a batch runs on them when one of its systems has a kicked or a massless pair,
so every batch here holds one of each beside systems of Kepler pairs: both row
updates, one and two systems a wave, whole runs and rounds with restarts, and
batches of which one class stays on one wave while the other divides its steps.
The reference row update gives the oracle's bits; the factored one re-associates
sums (1e-12 of the transit times, 1e-10 of an array's largest entry for the
gradients, as in test_gpu_row_update.py)."""
import numpy as np
import pytest

import oracle_lib as O
import nbodygradient_amd as nb
from nbodygradient_amd import workloads as W
from nbodygradient_amd.batch import Batch

pytestmark = pytest.mark.gpu

KEPLER, KICKED, MASSLESS = 0, 1, 2


def _systems(ns, kinds, seed, steps):
    """Specs, initial states and pair masks; a massless system starts from the
    state of its massive elements."""
    rng = np.random.default_rng(seed)
    specs, pairs = [], []
    for k, n in enumerate(ns):
        s = W.c2_system(rng, n)
        s.tmax = (steps + 7 * k) * s.h
        specs.append(s)
        pairs.append(np.zeros((n, n), dtype=np.uint8, order="F"))
    states = W.initial_states(specs, processes=1)
    for k, kind in enumerate(kinds):
        n = specs[k].n
        if kind == KICKED:
            pairs[k][n - 2, n - 1] = pairs[k][n - 1, n - 2] = 1
        if kind == MASSLESS:
            specs[k].elements = specs[k].elements.copy()
            specs[k].elements[n - 2:, 0] = 0.0
    return specs, states, pairs


def _run(specs, states, pairs, factored, perwave, rounds=None):
    ctx = nb.default_context()
    ctx.set_row_update(1 if factored else 0)
    ctx.set_systems_per_wave(perwave)
    ctx.set_grid_cap(2 if perwave == 2 else 0)  # few workgroups, so that systems are paired
    try:
        b = Batch(specs, states, pair=pairs)
        if rounds:
            for steps in rounds:
                st = b.round(steps, restart=False)
        else:
            st = b.run()
        res = b.download()
        b.close()
    finally:
        ctx.set_row_update(0)
        ctx.set_systems_per_wave(1)
        ctx.set_grid_cap(0)
    return st, res


def _close(a, b, rel):
    return a.shape == b.shape and (a.size == 0 or np.max(np.abs(a - b)) <= rel * np.max(np.abs(b)))


def _check(specs, states, pairs, res, factored):
    total = 0
    for s, (x, v, j), p, r in zip(specs, states, pairs, res):
        os_ = O.OState(x, v, s.elements[:, 0], t=s.t0, jac_init=j, pair=p)
        tt, dq, de, count = O.integrate_transits(os_, s.h, s.tmax, s.ntt(), grad=True)
        total += int(count.sum())
        assert np.array_equal(r["count"], count), s.n
        assert np.array_equal(r["x"], os_.x) and np.array_equal(r["v"], os_.v), s.n
        if factored:
            assert _close(r["tt"], tt, 1e-12) and _close(r["dtdq0"], dq, 1e-10) and _close(r["dtdelements"], de, 1e-10), s.n
        else:
            assert np.array_equal(r["tt"], tt), s.n
            assert np.array_equal(r["dtdq0"], dq) and np.array_equal(r["dtdelements"], de), s.n
    assert total > 0


@pytest.mark.parametrize("rounds", [None, (23, 23, 200)])
@pytest.mark.parametrize("perwave", [1, 2])
@pytest.mark.parametrize("factored", [False, True])
def test_kicked_and_massless_systems_in_a_class(factored, perwave, rounds):
    print("gpu: one wave, factored %d, %d a wave, rounds %s" % (factored, perwave, rounds), flush=True)
    ns = [9, 9, 9, 8, 8, 7, 7, 6, 6, 5, 5, 4, 4, 3, 3, 3, 2, 2, 8, 5]
    kinds = [KEPLER] * len(ns)
    kinds[2], kinds[18], kinds[15] = KICKED, MASSLESS, KICKED
    sys_ = _systems(ns, kinds, 900, 60)
    st, res = _run(*sys_, factored, perwave, rounds)
    assert (st["paired_systems"] > 0) == (perwave == 2)
    _check(*sys_, res, factored)


@pytest.mark.parametrize("factored", [False, True])
@pytest.mark.parametrize("perwave", [1, 2])
@pytest.mark.parametrize("large", [KICKED, MASSLESS, KEPLER])
def test_classes_on_different_launches(large, perwave, factored):
    # class 12 on one wave beside a class that divides its steps, or the reverse
    print("gpu: classes apart, kind %d, %d a wave, factored %d" % (large, perwave, factored), flush=True)
    ns = [12, 12, 11, 9, 9, 7, 7, 5, 5, 5, 3, 3, 3, 3]
    kinds = [KEPLER] * len(ns)
    if large == KEPLER:
        kinds[4], kinds[9] = KICKED, MASSLESS
    else:
        kinds[1] = large
    sys_ = _systems(ns, kinds, 910 + large, 50)
    _, res = _run(*sys_, factored, perwave)
    _check(*sys_, res, factored)
