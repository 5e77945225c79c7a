"""What is timed of this framework, and how: the work its users have it do.

Every case is one pass through a public entry point: single systems through
State / Integrator / TransitTiming (the reference's call pattern), batches and
rounds through Batch, requests through Server.  Systems are a star with
planets on nearly edge-on orbits, drawn as the benchmark workloads draw them
(periods log-uniform in [2, 200] d with neighbours at least 1.3 apart, masses
log-uniform in [1e-6, 3e-5], e < 0.05, h = P_in / 30).

`exact` restates the AHL21 map in plain numpy: every derivative by a complex
step (one column of the arrays per initial coordinate), transit times by
Newton's method on the map.
"""
import math
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nbodygradient.jl_amd"))

import nbodygradient_amd as nb  # noqa: E402
from nbodygradient_amd import _lib  # noqa: E402
from nbodygradient_amd.batch import Batch  # noqa: E402
from nbodygradient_amd.server import Server  # noqa: E402
from nbodygradient_amd.workloads import SystemSpec  # noqa: E402

GNEWT = 39.4845 / (365.242 * 365.242)  # AU^3 / (Msun d^2)
TWO_PI = 2.0 * math.pi
EPS = 1e-40  # the complex step


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one integrator step with its Jacobian from a host loop: the smallest call
        {"name": "step", "kind": "step", "n": 3, "steps": 1, "grad": True, "factored": False},
        # a plain orbit integration without derivatives (stability runs, plots)
        {"name": "orbit", "kind": "steps", "n": 5, "steps": 400, "grad": False, "factored": False},
        # state transition matrix over an arc
        {"name": "arc", "kind": "steps", "n": 9, "steps": 80, "grad": True, "factored": False},
        # trajectory output with the Jacobian before every step
        {"name": "trajectory", "kind": "trajectory", "n": 4, "steps": 150, "grad": True, "factored": False},
        # transit times and gradients of one system, as a fit that calls one system at a time does:
        # a small system over a whole observing season, and a long resonant chain
        {"name": "timing-3", "kind": "transits", "n": 3, "steps": 500, "ntbv": 1, "grad": True, "factored": False},
        {"name": "timing-8", "kind": "transits", "n": 8, "steps": 150, "ntbv": 1, "grad": True, "factored": True},
        # transit times, durations and depths (TransitParameters)
        {"name": "parameters-6", "kind": "transits", "n": 6, "steps": 150, "ntbv": 3, "grad": True, "factored": False},
        # a few walkers of a sampler, fewer than the card has room for
        {"name": "walkers", "kind": "fit", "n": 7, "systems": 61, "steps": 150, "ntbv": 1, "factored": False, "perwave": 1},
        # an ensemble of perturbed six-body systems, one run each
        {"name": "ensemble", "kind": "fit", "n": 6, "systems": 1024, "steps": 300, "ntbv": 1, "factored": False,
         "perwave": 1},
        # the survey batch in rounds, two systems per wave: factored Jacobian updates, and the reference's order
        {"name": "survey", "kind": "rounds", "n": 9, "systems": 4096, "steps": 250, "ntbv": 1, "factored": True,
         "perwave": 2},
        {"name": "survey-exact", "kind": "rounds", "n": 9, "systems": 2048, "steps": 200, "ntbv": 1, "factored": False,
         "perwave": 2},
        # requests of mixed size through the server until all are answered
        {"name": "serving", "kind": "serve", "n": 10, "systems": 96, "steps": 200, "ntbv": 1, "factored": False},
    ]


def _tmax(steps, h):
    """A run of `steps` steps: it ends a little before the last one does, so that the transit slots a run is given
    (the periods it spans, rounded up) depend on the steps alone."""
    return (steps - 0.25) * h


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "steps", "trajectory", "transits", "transits", "fit", "fit", "rounds", "rounds", "serve"])
    factored = rng.random() < 0.5
    ntbv = 3 if rng.random() < 0.25 else 1
    if kind == "step":
        return {"kind": kind, "n": rng.randint(2, 12), "steps": 1, "grad": rng.random() < 0.7, "factored": factored}
    if kind == "steps":
        return {"kind": kind, "n": rng.randint(2, 10), "steps": _log_int(rng, 10, 200), "grad": rng.random() < 0.7,
                "factored": factored}
    if kind == "trajectory":
        return {"kind": kind, "n": rng.randint(2, 8), "steps": _log_int(rng, 10, 150), "grad": rng.random() < 0.7,
                "factored": False}
    if kind == "transits":
        n = rng.randint(2, 10)
        return {"kind": kind, "n": n, "steps": _log_int(rng, 40, 1200 // n), "ntbv": ntbv, "grad": rng.random() < 0.8,
                "factored": factored}
    if kind == "serve":
        return {"kind": kind, "n": rng.randint(6, 10), "systems": _log_int(rng, 8, 96), "steps": _log_int(rng, 40, 200),
                "ntbv": ntbv, "factored": factored}
    n = rng.randint(3, 9)
    systems = _log_int(rng, 17, 4096)
    most = 250 if kind == "rounds" else 150
    steps = max(20, min(_log_int(rng, 30, most), 600000 // systems))
    return {"kind": kind, "n": n, "systems": systems, "steps": steps, "ntbv": ntbv, "factored": factored,
            "perwave": rng.randint(1, 2)}


# ------------------------------------------------------------------ inputs
def _periods(rng, k):
    while True:
        p = np.sort(np.exp(rng.uniform(math.log(2.0), math.log(200.0), k)))
        if k == 1 or np.all(p[1:] / p[:-1] >= 1.3):
            return p


def _elements(rng, n):
    """n x 7 rows (m, P, t0, e cos w, e sin w, I, Omega), the star first."""
    k = n - 1
    p = _periods(rng, k)
    e, w = rng.uniform(0.001, 0.05, k), rng.uniform(0.0, TWO_PI, k)
    el = np.zeros((n, 7))
    el[0, 0] = 1.0
    el[1:, 0] = np.exp(rng.uniform(math.log(1e-6), math.log(3e-5), k))
    el[1:, 1] = p
    el[1:, 2] = rng.uniform(0.0, 1.0, k) * p
    el[1:, 3], el[1:, 4] = e * np.cos(w), e * np.sin(w)
    el[1:, 5] = math.pi / 2 + rng.uniform(-0.01, 0.01, k)
    el[1:, 6] = rng.uniform(0.0, TWO_PI, k)
    return el


def _one(case, seed):
    """The elements and step of a single-system case."""
    el = _elements(np.random.default_rng(seed), case["n"])
    return el, el[1, 1] / 30.0


def _specs(case, seed):
    rng = np.random.default_rng(seed)
    steps = case["steps"]
    if case["kind"] == "fit":  # perturbations of one system, as a sampler draws them
        base = _elements(rng, case["n"])
        h = base[1, 1] / 30.0
        out = []
        for _ in range(case["systems"]):
            el = base.copy()
            k = case["n"] - 1
            el[1:, 0] *= 1.0 + 1e-4 * rng.standard_normal(k)
            el[1:, 1] *= 1.0 + 1e-5 * rng.standard_normal(k)
            el[1:, 3] *= 1.0 + 1e-3 * rng.standard_normal(k)
            el[1:, 4] *= 1.0 + 1e-3 * rng.standard_normal(k)
            out.append(SystemSpec(el, 0.0, h, _tmax(steps, h)))
        return out
    lo = 2 if case["kind"] == "serve" else 3
    out = []
    for i in range(case["systems"]):
        el = _elements(rng, lo + i % (case["n"] + 1 - lo))  # every body count as often
        h = el[1, 1] / 30.0
        # requests end at different times; a round advances every system by the same number of steps
        ns = steps // 4 + (37 * i) % (steps - steps // 4 + 1) if case["kind"] == "serve" else steps
        out.append(SystemSpec(el, 0.0, h, _tmax(ns, h)))
    return out


_contexts = {}


def _context(case):
    """The library context a program keeps for its settings."""
    key = (bool(case["factored"]), case.get("perwave", 1))
    if key not in _contexts:
        c = nb.Context()
        c.set_row_update(int(key[0]))
        c.set_systems_per_wave(key[1])
        _contexts[key] = c
    return _contexts[key]


class _Work:
    pass


def prepare(case, seed):
    w = _Work()
    w.kind, w.ctx, w.steps = case["kind"], _context(case), case["steps"]
    if w.kind in ("step", "steps", "trajectory", "transits"):
        el, w.h = _one(case, seed)
        ic = nb.ElementsIC(0.0, case["n"], el)
        w.start, w.s, w.grad = nb.State(ic), nb.State(ic), case["grad"]
        w.tmax = _tmax(w.steps, w.h)
        w.integrator = nb.Integrator(w.h, w.tmax)
        if w.kind == "transits":
            w.tt = (nb.TransitParameters if case["ntbv"] == 3 else nb.TransitTiming)(w.tmax, ic)
        if w.kind == "trajectory":
            w.out = nb.CartesianOutput(case["n"], w.steps, jacobian=w.grad)
        return w
    specs = _specs(case, seed)
    if w.kind == "serve":
        w.specs, w.ntbv = specs, case["ntbv"]
        b = Batch(specs, device_ic=True, ctx=w.ctx)
        w.states = b.initial()
        b.close()
        w.server = Server(max_bytes=2 << 30, chunk=64, ctx=w.ctx)
        return w
    w.batch = Batch(specs, ntbv=case["ntbv"], device_ic=True, ctx=w.ctx)
    nbod, ntt = w.batch.n.astype(np.int64), w.batch.ntt
    nb_ = case["ntbv"]
    # the arrays that a fit loop reads its results into
    w.tt = np.full(int((nb_ * nbod * ntt).sum()), 0.0)
    w.dq = np.full(int((nb_ * nbod ** 2 * 7 * ntt).sum()), 0.0)
    w.de = np.full(w.dq.size, 0.0)
    w.count = np.full(int(nbod.sum()), 0, dtype=np.int64)
    w.x, w.v = np.full(3 * w.count.size, 0.0), np.full(3 * w.count.size, 0.0)
    return w


# ------------------------------------------------------------------ one pass
def run(w):
    if w.kind == "step":
        w.s.set_state(w.start)
        if not w.grad:
            nb.ahl21(w.s, w.h, ctx=w.ctx)
            return {"x": w.s.x, "v": w.s.v}
        nb.ahl21(w.s, None, w.h, ctx=w.ctx)
        return {"x": w.s.x, "v": w.s.v, "jac": w.s.jac_step, "dqdt": w.s.dqdt}
    if w.kind == "steps":
        w.s.set_state(w.start)
        w.integrator(w.s, w.steps, grad=w.grad, ctx=w.ctx)
        if not w.grad:
            return {"x": w.s.x, "v": w.s.v}
        return {"x": w.s.x, "v": w.s.v, "jac": w.s.jac_step, "dqdt": w.s.dqdt}
    if w.kind == "trajectory":
        w.s.set_state(w.start)
        w.integrator(w.s, w.out, grad=w.grad, ctx=w.ctx)
        out = {"t": w.out.t, "x": w.out.x, "v": w.out.v}
        if w.grad:
            out["jac"] = w.out.jac_step
        return out
    if w.kind == "transits":
        w.s.set_state(w.start)
        w.tt.zero_out()
        w.integrator(w.s, w.tt, grad=w.grad, ctx=w.ctx)
        timing = isinstance(w.tt, nb.TransitTiming)
        out = {"count": w.tt.count, "tt": w.tt.tt if timing else w.tt.ttbv, "x": w.s.x, "v": w.s.v}
        if w.grad:
            out["dtdq0"] = w.tt.dtdq0 if timing else w.tt.dtbvdq0
            out["dtdelements"] = w.tt.dtdelements if timing else w.tt.dtbvdelements
            out["jac"] = w.s.jac_step
        return out
    if w.kind == "serve":
        ids = [w.server.submit(s, st, ntbv=w.ntbv) for s, st in zip(w.specs, w.states)]
        got = {}
        while len(got) < len(ids):
            w.server.step()
            for rid in w.server.finished():
                got[rid] = w.server.fetch(rid)
        return {k: np.concatenate([got[i][k].ravel(order="F") for i in ids])
                for k in ("tt", "dtdq0", "dtdelements", "count", "x", "v")}
    if w.kind == "fit":
        w.batch.reset()
        w.batch.run()
    else:
        w.batch.round(w.steps)  # systems that have ended start again
    rc = _lib.lib().nbg_batch_download(w.batch._h, _lib.dptr(w.tt), _lib.dptr(w.dq), _lib.dptr(w.de),
                                       _lib.i64ptr(w.count), _lib.dptr(w.x), _lib.dptr(w.v))
    w.ctx.check(rc, "nbg_batch_download")
    return {"tt": w.tt, "dtdq0": w.dq, "dtdelements": w.de, "count": w.count, "x": w.x, "v": w.v}


# ------------------------------------------------------------------ work
def _step_flops(n, grad):
    """One step: n (n - 1) Kepler drifts and the force-gradient correction; with the Jacobian each drift's 6 x 8
    derivative, 36 multiply-adds, the mass terms and compensated sums per column, and Phi * J."""
    f = n * (n - 1) * 700.0 + n * n * 60.0
    if grad:
        f += n * (n - 1) * (900.0 + 7 * n * (72 + 24 + 60)) + n * (n - 1) / 2 * 4 * n * 60.0 + 7 * n * (24.0 * n * n + 30 * n)
    return f


def _system_work(n, steps, ntt, ntbv, grad, transits):
    flops = (steps + (transits if grad else 0)) * _step_flops(n, grad) + 3.0 * transits * _step_flops(n, False)
    size = 8.0 * (24 * n + 1)  # the state in and out
    if grad:
        flops += 2.0 * transits * ntbv * (7 * n) ** 2
        size += 8.0 * 3 * 49 * n * n
    return flops, size + 8.0 * ntbv * n * ntt * (1 + (14 * n if grad else 0))


def work(case):
    n, steps, grad = case["n"], case["steps"], case.get("grad", True)
    # a typical system: its inner period is 30 steps, each planet twice the period of the one inside
    def transits(k):
        return sum(steps / (30.0 * 2.0 ** i) for i in range(k - 1))
    ntt = steps // 30 + 4
    if case["kind"] in ("step", "steps", "trajectory"):
        f, b = _system_work(n, steps, 0, 0, grad, 0)
        if case["kind"] == "trajectory":
            b += 8.0 * steps * (1 + 12 * n + (98 * n * n if grad else 0))
    elif case["kind"] == "transits":
        f, b = _system_work(n, steps, ntt, case["ntbv"], grad, transits(n))
    elif case["kind"] == "fit":
        f, b = [case["systems"] * q for q in _system_work(n, steps, ntt, case["ntbv"], True, transits(n))]
    else:
        lo = 2 if case["kind"] == "serve" else 3
        part = 0.625 if case["kind"] == "serve" else 1.0
        f = b = 0.0
        for k in range(lo, n + 1):
            fk, bk = _system_work(k, steps * part, ntt, case["ntbv"], True, part * transits(k))
            f += fk * case["systems"] / (n + 1 - lo)
            b += bk * case["systems"] / (n + 1 - lo)
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------ the exact results
def _sq(a):
    return (a * a).sum(-1)


def _angle(y, x):
    """atan2 with a complex step in its arguments."""
    return np.arctan2(y.real, x.real) + 1j * (x.real * y.imag - y.real * x.imag) / (x.real ** 2 + y.real ** 2)


def _cartesian(el):
    """Positions and velocities [.., n, 3] of element rows [.., n, 7] at time 0: each planet's Kepler orbit about
    the centre of mass of the bodies inside it, the whole system's centre of mass at rest in the origin."""
    n = el.shape[-2]
    m = el[..., 0]
    total = np.cumsum(m, axis=-1)
    r, v = np.zeros(el.shape[:-1] + (3,), dtype=complex), np.zeros(el.shape[:-1] + (3,), dtype=complex)
    for i in range(1, n):
        p, t0, ec, es, inc, om = (el[..., i, q] for q in range(1, 7))
        mean_motion = TWO_PI / p
        a = np.exp(np.log(GNEWT * total[..., i] * p * p / (4.0 * math.pi ** 2)) / 3.0)
        e = np.sqrt(ec * ec + es * es)
        root = np.sqrt(1.0 - e * e)
        tp = t0 - root / mean_motion * ec / (1.0 - es) - 2.0 / mean_motion * _angle(
            np.sqrt(1.0 - e) * (es + ec + e), np.sqrt(1.0 + e) * (es - ec - e))
        mean = -mean_motion * tp
        ecc = mean + e * np.sin(mean)
        for _ in range(12):
            ecc = ecc - (ecc - e * np.sin(ecc) - mean) / (1.0 - e * np.cos(ecc))
        c, s = np.cos(ecc), np.sin(ecc)
        rate = mean_motion / (1.0 - e * c)
        cw, sw = ec / e, es / e
        for dest, px, py in ((r, a * (c - e), a * root * s), (v, -a * rate * s, a * rate * root * c)):
            u, q = cw * px - sw * py, sw * px + cw * py
            q, z = np.cos(inc) * q, np.sin(inc) * q
            dest[..., i, 0] = np.cos(om) * u - np.sin(om) * q
            dest[..., i, 1] = np.sin(om) * u + np.cos(om) * q
            dest[..., i, 2] = z
    out = []
    for rel in (r, v):
        pos = np.zeros_like(rel)
        com = np.zeros(rel.shape[:-2] + (3,), dtype=complex)
        for i in range(n - 1, 0, -1):
            share = (m[..., i] / total[..., i])[..., None]
            pos[..., i, :] = com + (1.0 - share) * rel[..., i, :]
            com = com - share * rel[..., i, :]
        pos[..., 0, :] = com
        out.append(pos)
    return out


def _initial(el):
    """x, v [n, 3] and d (x, v, m) / d (P, t0, e cos w, e sin w, I, Omega, m), 7n x 7n, body by body."""
    n = el.shape[0]
    cols = np.repeat(el[None].astype(complex), 7 * n + 1, axis=0)
    for b in range(n):
        for k in range(7):
            if b > 0 or k == 6:
                cols[7 * b + k, b, (k + 1) % 7] += 1j * EPS
    x, v = _cartesian(cols)
    jac = np.zeros((7 * n, 7 * n))
    for b in range(n):
        for q in range(3):
            jac[7 * b + q] = x[:-1, b, q].imag / EPS
            jac[7 * b + 3 + q] = v[:-1, b, q].imag / EPS
        jac[7 * b + 6, 7 * b + 6] = 1.0
    return x[-1].real, v[-1].real, jac


def _kepler(x0, v0, k, h, drift_first):
    """The change of the relative coordinates by a drift of -h and a Kepler step of h (in that order, or the other)."""
    y = x0 - h[..., None] * v0 if drift_first else x0
    r0 = np.sqrt(_sq(y))
    beta = 2.0 * k / r0 - _sq(v0)
    eta = (y * v0).sum(-1)
    bound = beta.real > 0
    root = np.sqrt(np.where(bound, beta, -beta))
    s = h / r0
    for it in range(9):
        half = 0.5 * root * s
        sn, cs = np.where(bound, np.sin(half), np.sinh(half)), np.where(bound, np.cos(half), np.cosh(half))
        g1, g2 = 2.0 * sn * cs / root, 2.0 * sn * sn / (root * root)
        g3 = (s - g1) / beta
        r = r0 + eta * g1 + (k - r0 * beta) * g2
        if it < 8:
            s = s - (r0 * g1 + eta * g2 + k * g3 - h) / r
    fm1, gmh, fd, gdm1 = (q[..., None] for q in (-k * g2 / r0, -k * g3, -k * g1 / (r * r0), -k * g2 / r))
    dx, dv = fm1 * y + gmh * v0, fd * y + gdm1 * v0
    return (dx, dv) if drift_first else (dx - h[..., None] * dv, dv)


def _step(x, v, m, h):
    """One AHL21 step of every column: x, v [c, n, 3], m [c, n], h [c] (all complex)."""
    n = m.shape[1]
    x, v = x + 0.5 * h[:, None, None] * v, v.copy()
    pairs = [(i, j) for i in range(n - 1) for j in range(i + 1, n)]

    def sweep(order, drift_first):
        # pairs that share no body commute: take each run of such pairs at once
        level, levels = [0] * n, {}
        for i, j in order:
            at = max(level[i], level[j])
            level[i] = level[j] = at + 1
            levels.setdefault(at, []).append((i, j))
        for at in sorted(levels):
            i, j = [p[0] for p in levels[at]], [p[1] for p in levels[at]]
            mt = m[:, i] + m[:, j]
            dx, dv = _kepler(x[:, i] - x[:, j], v[:, i] - v[:, j], GNEWT * mt, np.repeat(0.5 * h[:, None], len(i), 1),
                             drift_first)
            wi, wj = (m[:, j] / mt)[..., None], (m[:, i] / mt)[..., None]
            x[:, i] += wi * dx
            x[:, j] -= wj * dx
            v[:, i] += wi * dv
            v[:, j] -= wj * dv

    sweep(pairs, True)
    i, j = [p[0] for p in pairs], [p[1] for p in pairs]
    rel = x[:, i] - x[:, j]
    r2 = _sq(rel)
    r1 = np.sqrt(r2)
    acc = np.zeros_like(x)
    pull = GNEWT * rel / (r2 * r1)[..., None]
    for p, (a, b) in enumerate(pairs):
        acc[:, a] -= m[:, b, None] * pull[:, p]
        acc[:, b] += m[:, a, None] * pull[:, p]
    da = acc[:, i] - acc[:, j]
    coeff = (h ** 3 / 24.0 * GNEWT)[:, None] / (r2 * r2 * r1)
    kick = coeff[..., None] * (rel * (2.0 * GNEWT * (m[:, i] + m[:, j]) / r1 + 3.0 * (da * rel).sum(-1))[..., None]
                               - r2[..., None] * da)
    for p, (a, b) in enumerate(pairs):
        v[:, a] += m[:, b, None] * kick[:, p]
        v[:, b] -= m[:, a, None] * kick[:, p]
    sweep(pairs[::-1], False)
    return x + 0.5 * h[:, None, None] * v, v


class _Orbit:
    """The columns of a system: one for each initial coordinate (x, v, m of each body), perturbed by the complex
    step, or a single real one without derivatives."""

    def __init__(self, el, h, grad):
        x, v, self.jinit = _initial(el)
        self.n, c = el.shape[0], 7 * el.shape[0] if grad else 1
        self.x, self.v = (np.repeat(q[None].astype(complex), c, axis=0) for q in (x, v))
        self.m = np.repeat(el[None, :, 0].astype(complex), c, axis=0)
        if grad:
            for b in range(self.n):
                for q in range(3):
                    self.x[7 * b + q, b, q] += 1j * EPS
                    self.v[7 * b + 3 + q, b, q] += 1j * EPS
                self.m[7 * b + 6, b] += 1j * EPS
        self.h = np.full(c, h, dtype=complex)
        self.one = np.zeros(1, dtype=complex)

    def go(self):
        self.before = self.x, self.v
        self.x, self.v = _step(self.x, self.v, self.m, self.h)

    def along(self, x, v, dt):
        """State after a step dt from (x, v), and its derivative by dt."""
        a, b = _step(x[:1].real + 0j, v[:1].real + 0j, self.m[:1].real + 0j, self.one + dt + 1j * EPS)
        return a[0].real, b[0].real, a[0].imag / EPS, b[0].imag / EPS

    def dqdt(self):
        _, _, a, b = self.along(*self.before, self.h[0].real)
        return np.concatenate([np.concatenate([a[i], b[i], [0.0]]) for i in range(self.n)])

    def jac(self):
        return np.asfortranarray(np.stack([np.concatenate([self.x[:, b], self.v[:, b], self.m[:, b, None]], axis=1)
                                           for b in range(self.n)], axis=1).reshape(7 * self.n, -1).imag.T / EPS)

    def xv(self):
        return self.x[0].real.T, self.v[0].real.T


def _exact_transits(case, o, h, el):
    n, grad, nb_ = case["n"], case["grad"], case["ntbv"]
    tmax = _tmax(case["steps"], h)
    ntt = int(np.max(np.ceil(np.abs(tmax / el[1:, 1]))) + 3)
    tt, dq = np.zeros((3, n, ntt)), np.zeros((3, n, ntt, 7 * n))
    count = np.zeros(n, dtype=np.int64)

    def sky(x, v, i):
        return ((x[i, :2] - x[0, :2]) * (v[i, :2] - v[0, :2])).sum()

    last = [sky(o.x[0].real, o.v[0].real, i) for i in range(n)]
    for step in range(case["steps"]):
        o.go()
        x, v = o.x[0].real, o.v[0].real
        for i in range(1, n):
            g = sky(x, v, i)
            if g > 0.0 and last[i] < 0.0 and -x[i, 2] > 0.25 * math.sqrt(_sq(x[i])):
                dt = -g * h / (g - last[i])
                for _ in range(7):
                    xt, vt, xd, vd = o.along(o.x, o.v, dt)
                    gd = ((xd[i, :2] - xd[0, :2]) * (vt[i, :2] - vt[0, :2])
                          + (xt[i, :2] - xt[0, :2]) * (vd[i, :2] - vd[0, :2])).sum()
                    dt -= sky(xt, vt, i) / gd
                dx, dv = xt[i, :2] - xt[0, :2], vt[i, :2] - vt[0, :2]
                c = count[i]
                count[i] += 1
                vsky = math.sqrt((dv * dv).sum())
                tt[:, i, c] = h * (step + 1) + dt, vsky, (dx * dx).sum()
                if grad:
                    xs, vs = _step(o.x, o.v, o.m, 0.0 * o.h + dt)
                    jx, jv = (xs[:, i, :2] - xs[:, 0, :2]).imag / EPS, (vs[:, i, :2] - vs[:, 0, :2]).imag / EPS
                    dq[0, i, c] = -((jx * dv).sum(-1) + (jv * dx).sum(-1)) / gd
                    dq[1, i, c] = ((jv * dv).sum(-1) + (dv * (vd[i, :2] - vd[0, :2])).sum() * dq[0, i, c]) / vsky
                    dq[2, i, c] = 2.0 * (jx * dx).sum(-1)
            last[i] = g
    x, v = o.xv()
    out = {"count": count, "tt": tt[0] if nb_ == 1 else tt, "x": x, "v": v}
    if grad:
        de = dq @ o.jinit
        for name, a in (("dtdq0", dq), ("dtdelements", de)):
            a = a.reshape(3, n, ntt, n, 7).transpose(0, 1, 2, 4, 3)
            out[name] = a[0] if nb_ == 1 else a
        out["jac"] = o.jac()
    return out


def exact(case, seed):
    if case["kind"] not in ("step", "steps", "trajectory", "transits"):
        return None  # hundreds of systems: more than this takes in seconds
    if case["grad"] and case["steps"] * case["n"] ** 2 > 12000 and case["n"] > 3:
        return None
    el, h = _one(case, seed)
    o = _Orbit(el, h, case["grad"])
    if case["kind"] == "transits":
        return _exact_transits(case, o, h, el)
    if case["kind"] == "trajectory":
        n, ns = case["n"], case["steps"]
        out = {"t": h * np.arange(ns), "x": np.zeros((3, n, ns)), "v": np.zeros((3, n, ns))}
        if case["grad"]:
            out["jac"] = np.zeros((7 * n, 7 * n, ns))
        for k in range(ns):
            out["x"][..., k], out["v"][..., k] = o.xv()
            if case["grad"]:
                out["jac"][..., k] = o.jac()
            o.go()
        return out
    for _ in range(case["steps"]):
        o.go()
    x, v = o.xv()
    out = {"x": x, "v": v}
    if case["grad"]:
        out["jac"], out["dqdt"] = o.jac(), o.dqdt()
    return out
