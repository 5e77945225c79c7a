"""Cooperative workgroups forced beside two systems per wave: the cooperative
systems come off the front of each class's queue, and what is left runs by
units of one or two systems or, where the class forms no pair (a batch no
larger than the GPU's wave slots, bodies that are never paired), one by one.
Every system is integrated exactly once, so every output is the bits of the
default launch, which test_gpu_waves.py compares with the oracle."""
import numpy as np
import pytest

import nbodygradient_amd as nb
from nbodygradient_amd import workloads as W
from nbodygradient_amd.batch import Batch

pytestmark = pytest.mark.gpu


def _specs(ns, seed, steps=60):
    rng = np.random.default_rng(seed)
    out = []
    for k, n in enumerate(ns):
        s = W.c2_system(rng, n)
        s.tmax = (steps + k % 11) * s.h
        out.append(s)
    return out


def _run(specs, states, coop, perwave, rounds):
    ctx = nb.default_context()
    ctx.set_coop(*coop)
    ctx.set_systems_per_wave(perwave)
    try:
        b = Batch(specs, states)
        if rounds:
            st = [b.round(40, restart=False) for _ in range(2)][0]
        else:
            st = b.run()
        res = b.download(derivatives=True)
        b.close()
    finally:
        ctx.set_coop(1, 128)
        ctx.set_systems_per_wave(1)
    return st, res


@pytest.mark.parametrize("rounds", [False, True])
@pytest.mark.parametrize("ns,copies,most", [
    ([6], 200, 64),          # a compute unit each: the wide launch
    ([3, 6, 8], 110, 64),    # more systems than compute units, no pair formed
    ([9, 11, 12], 20, 5),    # classes that never pair
    ([4, 5], 1, 2),          # every system cooperative: nothing left over
    ([3, 5, 7], 700, 16),    # more systems than wave slots: pairs beside cooperative systems
])
def test_cooperative_systems_beside_two_per_wave(ns, copies, most, rounds):
    print("gpu: coop and two per wave, n=%s x %d, rounds %d" % (ns, copies, rounds), flush=True)
    specs = _specs(ns * min(copies, 5), 600 + len(ns))
    copies = max(1, copies // 5)
    states = W.initial_states(specs, processes=1)
    want = _run(specs, states, (1, 128), 1, rounds)[1]
    st, got = _run(specs * copies, states * copies, (2, most), 2, rounds)
    assert 0 < st["launches"][1]["grid"] <= most
    assert (st["paired_systems"] > 0) == (copies * len(specs) > 2048)
    for k, r in enumerate(got):
        w = want[k % len(specs)]
        for key in ("count", "tt", "dtdq0", "dtdelements", "x", "v"):
            assert np.array_equal(r[key], w[key]), (k, key)
