"""The launches that give a system two or three waves (nbg_split.h) against
the oracle: every body count, both row updates, every run mode they take, few
systems (three waves), many (two waves, the Jacobian in LDS or in HBM) and
pairs of systems, at odd counts and unequal run lengths.  The reference row
update is the oracle's arithmetic in the oracle's order, so its outputs are
the oracle's bits; the factored one re-associates sums, whose results may
differ by the 1e-10 (Jacobians) and 1e-12 (transit times) of an array's
largest entry that test_gpu_row_update.py asks for."""
import numpy as np
import pytest

import oracle_lib as O
import nbodygradient_amd as nb
from nbodygradient_amd import workloads as W
from nbodygradient_amd.batch import Batch, cartesian_batch

pytestmark = pytest.mark.gpu

NS = list(range(2, 13))


def _specs(n, count, seed, steps=70):
    rng = np.random.default_rng(seed)
    out = []
    for k in range(count):
        s = W.c2_system(rng, n)
        s.tmax = (steps + 13 * k) * s.h
        out.append(s)
    return out


def _close(a, b, rel):
    return a.shape == b.shape and (a.size == 0 or np.max(np.abs(a - b)) <= rel * np.max(np.abs(b)))


def _check(specs, states, res, grad, ntbv, factored):
    for s, (x, v, j), r in zip(specs, states, res):
        os_ = O.OState(x, v, s.elements[:, 0], t=s.t0, jac_init=j)
        o = O.integrate_transits(os_, s.h, s.tmax, s.ntt(), grad=grad, ntbv=ntbv)
        tt, count = o[0], o[-1]
        assert np.array_equal(r["x"], os_.x) and np.array_equal(r["v"], os_.v)
        assert np.array_equal(r["count"], count)
        if factored:
            assert _close(r["tt"], tt, 1e-12)
            assert _close(r["dtdq0"], o[1], 1e-10) and _close(r["dtdelements"], o[2], 1e-10)
        else:
            assert np.array_equal(r["tt"], tt)
            if grad:
                assert np.array_equal(r["dtdq0"], o[1]) and np.array_equal(r["dtdelements"], o[2])


def _run(specs, grad=True, ntbv=1, factored=False, perwave=1, cap=0, copies=1):
    ctx = nb.default_context()
    ctx.set_row_update(1 if factored else 0)
    ctx.set_systems_per_wave(perwave)
    ctx.set_grid_cap(cap)
    try:
        states = W.initial_states(specs, processes=1)
        b = Batch(specs * copies, states * copies, grad=grad, ntbv=ntbv)
        st = b.run()
        res = b.download(derivatives=grad)
        b.close()
    finally:
        ctx.set_row_update(0)
        ctx.set_systems_per_wave(1)
        ctx.set_grid_cap(0)
    if perwave == 2 and specs[0].n <= 7:
        assert st["paired_systems"] > 0
    assert len(res) == len(specs) * copies
    k = len(specs) * (copies - 1)
    _check(specs, states, res[:len(specs)], grad, ntbv, factored)
    if copies > 1:  # the last systems of the batch
        _check(specs, states, res[k:], grad, ntbv, factored)


@pytest.mark.parametrize("form", ["reference", "factored", "three observables", "no gradient"])
@pytest.mark.parametrize("n", NS)
def test_three_waves(n, form):
    print("gpu: three waves n=%d %s" % (n, form), flush=True)
    _run(_specs(n, 3, 100 + n), grad=form != "no gradient", ntbv=3 if form == "three observables" else 1,
         factored=form == "factored")


@pytest.mark.parametrize("factored", [False, True])
@pytest.mark.parametrize("n", NS)
def test_two_waves(n, factored):
    # more systems than compute units
    print("gpu: two waves n=%d factored %d" % (n, factored), flush=True)
    _run(_specs(n, 3, 200 + n, 40), factored=factored, copies=101)


@pytest.mark.parametrize("factored", [False, True])
@pytest.mark.parametrize("n", NS)
def test_pairs(n, factored):
    # an odd count on a grid of two workgroups; bodies > 7 are never paired
    print("gpu: pairs n=%d factored %d" % (n, factored), flush=True)
    _run(_specs(n, 7, 250 + n, 40), factored=factored, perwave=2, cap=2)


@pytest.mark.parametrize("perwave,copies,cap", [(1, 9, 0), (2, 1, 3)])
def test_two_waves_mixed(perwave, copies, cap):
    print("gpu: two waves, mixed body counts, %d systems a workgroup" % perwave, flush=True)
    specs = [s for n in (2, 3, 5, 6, 7, 9, 10) for s in _specs(n, 5, 300 + n, 30)]
    _run(specs, perwave=perwave, copies=copies, cap=cap)


@pytest.mark.parametrize("n", [2, 5, 8, 12])
@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("frac", [0.0, 0.4])
def test_plain_run(n, grad, frac):
    # frac: a last short step onto the time
    print("gpu: plain run n=%d grad %d" % (n, grad), flush=True)
    s = _specs(n, 1, 400 + n)[0]
    ic = nb.ElementsIC(s.t0, n, s.elements)
    st = nb.State(ic)
    os_ = O.OState(st.x.copy(), st.v.copy(), s.elements[:, 0], t=s.t0)
    end = s.t0 + (37 + frac) * s.h
    nb.Integrator(s.h, s.t0, end)(st, end, grad=grad)
    O.integrate_to(os_, s.h, end, grad=grad)
    for k in ("x", "v") + (("jac_step", "jac_error", "dqdt") if grad else ()):
        assert np.array_equal(getattr(st, k), getattr(os_, k)), k


@pytest.mark.parametrize("n", [2, 4, 9, 12])
@pytest.mark.parametrize("copies", [1, 101])
def test_trajectories(n, copies):
    print("gpu: trajectories n=%d, %d systems" % (n, 3 * copies), flush=True)
    specs, N = _specs(n, 3, 500 + n), [5, 9, 2]
    states = W.initial_states(specs, processes=1)
    got = cartesian_batch(specs * copies, N * copies, states=states * copies, jacobian=True)
    for s, k, (x, v, j), r in zip(specs, N, states, got[-3:]):
        os_ = O.OState(x, v, s.elements[:, 0], t=s.t0, jac_init=j)
        rec = O.cartesian_output(os_, s.h, s.tmax, k)
        for key in ("t", "x", "v", "xerror", "verror", "jac_step", "jac_error"):
            assert np.array_equal(r[key], rec[key]), key
