"""Bounded waits between the waves of a workgroup (nbg_split.h).  With every
wait bounded to a single poll, a run on each of the launches -- a compute unit a
system, more systems than compute units, two systems a workgroup -- ends and
reports the failure, and the next one, with the default bounds, gives the usual
results.  A wave that has nothing to do for a whole run (no gradient, no
transit) does not run out of its bound while the state wave steps on.  The bound
is one on transit runs with cooperative workgroups allowed: others never had it."""
import numpy as np
import pytest

import oracle_lib as O
import nbodygradient_amd as nb
from nbodygradient_amd import workloads as W
from nbodygradient_amd.batch import Batch, cartesian_batch

pytestmark = pytest.mark.gpu


def _specs(ns, seed, steps):
    rng = np.random.default_rng(seed)
    out = []
    for n in ns:
        s = W.c2_system(rng, n)
        s.tmax = steps * s.h
        out.append(s)
    return out


def _run(specs, states, grad=True):
    b = Batch(specs, states, grad=grad)
    try:
        b.run()
        return b.download(derivatives=grad)
    finally:
        b.close()


def _check(spec, state, r, grad):
    x, v, j = state
    os_ = O.OState(x, v, spec.elements[:, 0], t=spec.t0, jac_init=j)
    o = O.integrate_transits(os_, spec.h, spec.tmax, spec.ntt(), grad=grad)
    assert np.array_equal(r["count"], o[-1]) and np.array_equal(r["tt"], o[0])
    assert np.array_equal(r["x"], os_.x) and np.array_equal(r["v"], os_.v)
    if grad:
        assert np.array_equal(r["dtdq0"], o[1]) and np.array_equal(r["dtdelements"], o[2])


@pytest.mark.parametrize("ns,copies,perwave,cap", [
    ([3, 9, 12], 1, 1, 0),      # three waves
    ([4, 6], 150, 1, 0),        # two waves, more systems than compute units
    ([8, 11], 150, 1, 0),       # ... the Jacobian in HBM
    ([3, 5, 7], 4, 2, 2),       # two systems a workgroup
])
def test_a_wait_that_runs_out_is_an_error(ns, copies, perwave, cap):
    print("gpu: wait bound, n=%s x %d, %d a workgroup" % (ns, copies, perwave), flush=True)
    specs = _specs(ns, 800, 70)
    states = W.initial_states(specs, processes=1)
    ctx = nb.default_context()
    ctx.set_systems_per_wave(perwave)
    ctx.set_grid_cap(cap)
    try:
        ctx.set_coop_wait(1)
        try:
            with pytest.raises(nb.NbgError) as ei:
                _run(specs * copies, states * copies)
            assert "timed out" in str(ei.value)
        finally:
            ctx.set_coop_wait(0)
        res = _run(specs * copies, states * copies)
    finally:
        ctx.set_systems_per_wave(1)
        ctx.set_grid_cap(0)
    for q, s in enumerate(specs):
        _check(s, states[q], res[q], True)
        _check(s, states[q], res[len(res) - len(specs) + q], True)


@pytest.mark.parametrize("copies", [1, 100])
def test_a_run_without_work_for_a_wave_is_no_failure(copies):
    # 4000 steps, some 0.1 s, against a bound of 2^16 polls, about 5 ms: no
    # planet transits in this tenth of the inner orbit
    print("gpu: waits of a whole run, %d copies" % copies, flush=True)
    specs = _specs([2, 3, 4], 810, 1)
    for s in specs:
        P = s.elements[1:, 1]
        s.elements[1:, 2] = -0.25 * P
        s.h = P[0] / 40000
        s.tmax = 4000 * s.h
    states = W.initial_states(specs, processes=1)
    ctx = nb.default_context()
    ctx.set_coop_wait(1 << 16)
    try:
        res = _run(specs * copies, states * copies, grad=False)
    finally:
        ctx.set_coop_wait(0)
    for q, s in enumerate(specs):
        _check(s, states[q], res[q], False)
        assert res[q]["count"].sum() == 0


def test_other_runs_are_not_bounded():
    print("gpu: a wait bound and runs it does not reach", flush=True)
    spec = _specs([4], 820, 60)[0]
    (x, v, j), = W.initial_states([spec], processes=1)
    ctx = nb.default_context()
    ctx.set_coop_wait(1)
    try:
        st = nb.State(nb.ElementsIC(spec.t0, spec.n, spec.elements))
        os_ = O.OState(st.x.copy(), st.v.copy(), spec.elements[:, 0], t=spec.t0)
        end = spec.t0 + 10 * spec.h
        nb.Integrator(spec.h, spec.t0, end)(st, end, grad=True)
        O.integrate_to(os_, spec.h, end, grad=True)
        for k in ("x", "v", "jac_step", "jac_error", "dqdt"):
            assert np.array_equal(getattr(st, k), getattr(os_, k)), k
        got = cartesian_batch([spec], [7], states=[(x, v, j)], jacobian=True)[0]
        os_ = O.OState(x, v, spec.elements[:, 0], t=spec.t0, jac_init=j)
        rec = O.cartesian_output(os_, spec.h, spec.tmax, 7)
        assert np.array_equal(got["x"], rec["x"]) and np.array_equal(got["jac_step"], rec["jac_step"])
        ctx.set_coop(0, 0)  # no cooperative workgroups, no bound
        _check(spec, (x, v, j), _run([spec], [(x, v, j)])[0], True)
    finally:
        ctx.set_coop(1, 128)
        ctx.set_coop_wait(0)
