"""Per-launch figures of a batch: a launch that took every class is the one
entry with a grid, a time and the work of all body counts; classes that ran no
launch of their own have zeros."""
import ctypes as C

import numpy as np
import pytest

from nbodygradient_amd import _lib
from nbodygradient_amd import workloads as W
from nbodygradient_amd.batch import Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [1, 100])
def test_one_entry_a_launch(copies):
    print("gpu: launch figures, %d copies" % copies, flush=True)
    rng = np.random.default_rng(830)
    ns = [5, 9, 10, 12]
    specs = [W.c2_system(rng, n) for n in ns]
    for s in specs:
        s.tmax = 20 * s.h
    b = Batch(specs * copies, W.initial_states(specs, processes=1) * copies)
    st = _lib.BatchStats()
    b.ctx.check(_lib.lib().nbg_batch_run(b._h, C.byref(st)), "nbg_batch_run")
    b.close()
    launched = [c for c in range(13) if st.launch_ms[c] > 0]
    # 4 systems: a compute unit each, one launch for all; 400: a launch a class
    assert launched == ([12] if copies == 1 else [9, 10, 12])
    for c in range(13):
        assert (st.launch_grid[c] > 0) == (c in launched)
        assert c in launched or sum(st.launch_units[c]) == 0
    assert sum(st.launch_units[c][n] for c in range(13) for n in range(2, 13)) == st.system_steps
