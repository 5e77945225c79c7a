"""A single system's record goes to the GPU and back in one piece; transit
outputs up to 1 MiB travel in it, larger ones by themselves.  Both sides of
that line, with and without gradients and with three observables: the oracle's
bits where transits were recorded, the caller's contents everywhere else, and
the same from a second call whose record is smaller."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from nbodygradient_amd import _lib, workloads as W
from nbodygradient_amd._lib import dptr, i64ptr, u8ptr
from nbodygradient_amd.ics import ElementsIC, init_nbody

pytestmark = pytest.mark.gpu

LINE = 1 << 20  # bytes of transit outputs


def _call(spec, grad, ntbv, ntt):
    n = spec.n
    x, v, jinit = init_nbody(ElementsIC(spec.t0, n, spec.elements))
    x, v, jinit = (np.asfortranarray(a) for a in (x, v, jinit))
    given = np.asfortranarray(np.random.default_rng(3).standard_normal((ntbv, n, ntt)))
    given_d = np.asfortranarray(np.random.default_rng(4).standard_normal((ntbv, n, ntt, 7, n)))
    r = {"x": x.copy(order="F"), "v": v.copy(order="F"), "J": np.asfortranarray(np.eye(7 * n)),
         "JE": np.zeros((7 * n, 7 * n), order="F"), "dqdt": np.zeros(7 * n), "tt": given.copy(order="F"),
         "dq": given_d.copy(order="F"), "de": given_d.copy(order="F"), "count": np.full(n, 7, dtype=np.int64)}
    t, z = C.c_double(spec.t0), np.zeros((3, n), order="F")
    ctx = _lib.default_context()
    rc = _lib.lib().nbg_integrate_transits(
        ctx.handle, n, C.c_double(spec.h), C.c_double(spec.tmax), 0, int(grad), ntbv, C.byref(t), dptr(r["x"]),
        dptr(r["v"]), dptr(z), dptr(z.copy(order="F")), dptr(np.ascontiguousarray(spec.elements[:, 0])),
        u8ptr(np.zeros((n, n), dtype=np.uint8, order="F")), dptr(r["J"]), dptr(r["JE"]), dptr(r["dqdt"]), dptr(jinit),
        C.c_int64(ntt), dptr(r["tt"]), dptr(r["dq"]), dptr(r["de"]), i64ptr(r["count"]))
    ctx.check(rc, "nbg_integrate_transits")
    os_ = O.OState(x, v, spec.elements[:, 0], t=spec.t0, jac_init=jinit)
    o = O.integrate_transits(os_, spec.h, spec.tmax, spec.ntt(), grad=grad, ntbv=ntbv)
    assert np.array_equal(r["count"], o[-1]) and np.array_equal(r["x"], os_.x) and np.array_equal(r["v"], os_.v)
    assert o[-1].max() > 1
    if grad:
        assert np.array_equal(r["J"], os_.jac_step)
    k = spec.ntt()
    written = np.arange(k)[None, :] < o[-1][:, None]  # body, transit
    outs = [(r["tt"], given, o[0].reshape((ntbv, n, k), order="F"))]
    if grad:
        outs += [(r["dq"], given_d, o[1].reshape((ntbv, n, k, 7, n), order="F")),
                 (r["de"], given_d, o[2].reshape((ntbv, n, k, 7, n), order="F"))]
    else:
        assert np.array_equal(r["dq"], given_d) and np.array_equal(r["de"], given_d)
    for got, before, want in outs:
        mask = written.reshape((1, n, k) + (1,) * (got.ndim - 3))
        assert np.array_equal(got[:, :, :k], np.where(mask, want, before[:, :, :k]))
        assert np.array_equal(got[:, :, k:], before[:, :, k:])


@pytest.mark.parametrize("n,grad,ntbv", [(2, True, 1), (3, True, 3), (5, True, 1), (12, True, 1), (3, False, 1), (4, False, 3)])
def test_outputs_on_both_sides_of_the_line(n, grad, ntbv):
    print("gpu: single record n=%d grad=%s ntbv=%d" % (n, grad, ntbv), flush=True)
    spec = W.c2_system(np.random.default_rng(90 + n), n)
    spec.tmax = 95 * spec.h
    each = 8 * ntbv * n * ((1 + 14 * n) if grad else 1)
    last = LINE // each
    for ntt in (last, last + 1, spec.ntt()):
        _call(spec, grad, ntbv, ntt)
