"""Single steps of random states, bit for bit the oracle's: elliptic orbits of
every eccentricity, hyperbolic and nearly radial ones, steps from a thousandth of
a period to several, forward and backward, masses over six decades.  Neighbouring
pairs of one system mix the kinds, so the waves of a level hold lanes inside and
outside the common case of the Kepler solve (nbg_pair.h), whose quotients and
roots replace the compiler's.  Where a Jacobian overflows, the oracle's dense
products spread the NaN to entries the kernels leave alone (0 x NaN, mass rows
included): there the launch that divides a step between waves is compared
with the one-wave launch, entry by entry."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from nbodygradient_amd import _lib
from nbodygradient_amd._lib import dptr, i64ptr, u8ptr

pytestmark = pytest.mark.gpu


def _state(rng, n, kind):
    m = 10 ** rng.uniform(-6, 0, n)
    m[0] = 1.0
    x, v = np.zeros((3, n)), np.zeros((3, n))
    for i in range(1, n):
        r = 10 ** rng.uniform(-1, 1)
        d = rng.standard_normal(3)
        d /= np.linalg.norm(d)
        t = rng.standard_normal(3)
        t -= t @ d * d
        t /= np.linalg.norm(t)
        vc = np.sqrt(O.GNEWT / r)
        f = rng.uniform(0.9, 1.1) if kind == "circular" else 10 ** rng.uniform(-1.5, 0.7)
        a = 0.0 if kind == "circular" else rng.uniform(0, np.pi)
        x[:, i] = r * d
        v[:, i] = vc * f * (np.cos(a) * t + np.sin(a) * d)
    return np.asfortranarray(x), np.asfortranarray(v), m


def _transit_step(fn, n, x, v, m, h):
    g = [x.copy(order="F"), v.copy(order="F"), np.zeros((3, n), order="F"), np.zeros((3, n), order="F"),
         np.asfortranarray(np.eye(7 * n)), np.zeros((7 * n, 7 * n), order="F"), np.zeros(7 * n)]
    tt, dq = np.zeros((n, 2), order="F"), np.zeros((n, 2, 7, n), order="F")
    de, count, t = dq.copy(order="F"), np.zeros(n, dtype=np.int64), C.c_double(0.0)
    ctx = _lib.default_context()
    rc = fn(ctx.handle, n, C.c_double(abs(h)), C.c_double(h), 0, 1, 1, C.byref(t), *[dptr(a) for a in g[:4]], dptr(m),
            u8ptr(np.zeros((n, n), dtype=np.uint8, order="F")), *[dptr(a) for a in g[4:]],
            dptr(np.asfortranarray(np.eye(7 * n))), C.c_int64(2), dptr(tt), dptr(dq), dptr(de), i64ptr(count))
    ctx.check(rc, "transit step")
    return g + [tt, dq, de, count]


@pytest.mark.parametrize("kind", ["circular", "any"])
@pytest.mark.parametrize("n", [2, 3, 5, 8, 12])
def test_random_single_steps(n, kind):
    print("gpu: random states n=%d %s" % (n, kind), flush=True)
    rng = np.random.default_rng(1000 + n)
    ctx = _lib.default_context()
    pair = np.zeros((n, n), dtype=np.uint8, order="F")
    for _ in range(40):
        x, v, m = _state(rng, n, kind)
        rmin = np.min(np.linalg.norm(x[:, 1:], axis=0))
        period = 2 * np.pi * np.sqrt(rmin ** 3 / O.GNEWT)
        h = period * 10 ** rng.uniform(-3, -1.3 if kind == "circular" else 0.5) * rng.choice([-1.0, 1.0])
        os_ = O.OState(x, v, m)
        O.step(os_, h, grad=True)
        g = {"x": x.copy(order="F"), "v": v.copy(order="F"), "xe": np.zeros((3, n), order="F"),
             "ve": np.zeros((3, n), order="F"), "J": np.asfortranarray(np.eye(7 * n)),
             "JE": np.zeros((7 * n, 7 * n), order="F"), "q": np.zeros(7 * n)}
        rc = _lib.lib().nbg_ahl21_step(ctx.handle, n, C.c_double(h), 1, dptr(g["x"]), dptr(g["v"]), dptr(g["xe"]),
                                       dptr(g["ve"]), dptr(m), u8ptr(pair), dptr(g["J"]), dptr(g["JE"]), dptr(g["q"]))
        ctx.check(rc, "nbg_ahl21_step")
        finite = True
        for key, want in (("x", os_.x), ("v", os_.v), ("xe", os_.xerror), ("ve", os_.verror), ("J", os_.jac_step),
                          ("JE", os_.jac_error), ("q", os_.dqdt)):
            ok = np.isfinite(want)
            finite = finite and bool(ok.all())
            assert np.array_equal(g[key][ok], want[ok]), (key, h)
        if not finite:
            L = _lib.lib()
            three = _transit_step(L.nbg_integrate_transits, n, x, v, m, h)
            one = _transit_step(L.nbg_integrate_transits_noalloc, n, x, v, m, h)  # the one-wave launch
            for a, b in zip(three, one):
                assert np.array_equal(a, b, equal_nan=True), h
