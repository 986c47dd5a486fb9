"""The autotuner where the levels of a batch share a launch: the trials time
the shared launch (one time for both levels), the pick keeps both levels on one
block and depth, so that a tuned batch still shares, and the trials' steps are
ordinary ones. Timed steps afterwards have a launch per level again.
"""
from __future__ import annotations

import numpy as np
import pytest

from twoscalesplit_amd import MODE_BAND, MODE_PLAIN, MODE_REFERENCE, Solver, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,cap,density,force", [
    (MODE_REFERENCE, 60000, True, True), (MODE_BAND, 60000, True, True),
    (MODE_BAND, 262145, True, False), (MODE_REFERENCE, 262145, False, False),
    # the trials run with one lane per target, whatever the batch takes
    (MODE_REFERENCE, 720, True, True), (MODE_PLAIN, 60000, False, False)])
def test_shared_levels_get_one_shape(mode, cap, density, force):
    sc = scenes.small_two_scale(nx=24, ny=30, mode=mode, split_x=0.05)
    print("[case]", mode, cap, flush=True)
    a = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    b = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    try:
        r = a.autotune(1, 2)
        log = np.array([row[4:8] for row in r["trials"]])
        assert len(log) == 28
        t = a.get_tuning()
        for on, low in ((density, 0), (force, 2)):
            assert (log[:, low] == log[:, low + 1]).all() == on
            if on:
                assert t.block[low] == t.block[low + 1] and t.depth[low] == t.depth[low + 1]
        a.step_graph(4)
        b.step(r["steps_taken"])
        b.step_graph(4)
        for f in ("POS_L", "VEL_L", "RHO_L", "POS_H", "VEL_H", "RHO_H", "LIST_L", "LIST_H"):
            np.testing.assert_array_equal(a.read(f), b.read(f), err_msg=f)
        a.enable_timing(True)
        a.step(2)
        a.step_graph(2)
        assert len(a.phase_times()) == 8
    finally:
        a.close()
        b.close()


def test_refused_autotune_changes_nothing():
    """A state that host writes left invalid stops the autotuner's first step:
    timing, shapes and lanes stay as they were."""
    sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_BAND)
    sol = Solver(sc.cfg, sc.low_xy, 720, sc.bnd_xy)
    try:
        sol.step(1)
        lanes, shapes = sol.lanes(), sol.get_tuning().as_dict()
        sol.enable_timing(True)
        state = sol.read("STATE_L")
        bad = state.copy()
        bad[sol.read("LIST_L")[:1]] = 2
        sol.write("STATE_L", bad)
        with pytest.raises(RuntimeError, match="deleted particle listed"):
            sol.autotune(1, 1)
        assert sol.lanes() == lanes and sol.get_tuning().as_dict() == shapes
        sol.write("STATE_L", state)
        sol.step(2)
        assert all(v > 0 for v in sol.phase_times().values())
    finally:
        sol.close()
