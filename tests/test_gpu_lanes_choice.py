"""The choice of lanes per target: by the targets to expect, off once launch
shapes are set, back with reset_tuning, and the same after the autotuner as
before it. Results are the same throughout.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from twoscalesplit_amd import MODE_BAND, MODE_PLAIN, MODE_REFERENCE, Batch, Solver, _native as N, scenes

FIELDS = ("POS_L", "VEL_L", "RHO_L", "POS_H", "RHO_H", "LIST_L", "LIST_H", "LIST_G")


def test_null_arguments_are_refused():
    L, n = N.lib(), C.c_int()
    assert L.tss_reset_tuning(None) == L.tss_batch_reset_tuning(None) != N.TSS_OK
    assert L.tss_get_lanes(None, C.byref(n)) == L.tss_batch_get_lanes(None, C.byref(n)) != N.TSS_OK


@pytest.mark.gpu
@pytest.mark.parametrize("cap,lanes", [(720, 8), (30000, 4), (60000, 1)])
def test_set_and_reset(cap, lanes):
    sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_BAND)
    print("[case]", cap, lanes, flush=True)
    a = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    b = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    try:
        assert a.lanes() == b.lanes() == lanes
        default = b.get_tuning().as_dict()
        for k, t in enumerate((b.get_tuning(), N.TssTuning.uniform(128, 8, 1, 64))):
            a.step(2)
            a.step_graph(4)
            b.set_tuning(t)
            assert b.lanes() == 1
            b.step(2)
            b.reset_tuning()
            assert b.lanes() == lanes and b.get_tuning().as_dict() == default
            b.step_graph(4)
            for f in FIELDS:
                np.testing.assert_array_equal(a.read(f), b.read(f), err_msg=f"{f} {k}")
        b.autotune(1, 1)
        assert b.lanes() == lanes
        b.set_tuning(b.get_tuning())
        b.autotune(1, 1)
        assert b.lanes() == 1
    finally:
        a.close()
        b.close()


@pytest.mark.gpu
def test_batch():
    sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_BAND)
    b = Batch(2, 60000, 2 * len(sc.bnd_xy), 2 * sc.cells[0], 2 * sc.cells[1])
    try:
        one = b.add_scene(sc.cfg, sc.low_xy, 16000, sc.bnd_xy)
        assert b.lanes() == 8
        two = b.add_scene(sc.cfg, sc.low_xy, 16000, sc.bnd_xy)
        assert b.lanes() == 4
        b.set_tuning(N.TssTuning.uniform())
        assert b.lanes() == 1
        b.remove_scene(two)
        assert b.lanes() == 1
        b.reset_tuning()
        assert b.lanes() == 8
        b.step(3)
        assert b.counts(one)["step"] == 3
    finally:
        b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("mode,split_x,last", [
    (MODE_PLAIN, 0.0, (16384, 49152)), (MODE_BAND, -1.0, (16384, 49152)),
    (MODE_REFERENCE, 0.1, (5461, 16384)),
    # all split: the plane lies before the domain or on its edge
    (MODE_REFERENCE, 0.0, (5461, 12288)), (MODE_REFERENCE, -1.0, (5461, 12288))])
def test_lines(mode, split_x, last):
    """The capacities up to which a scene takes eight and four lanes."""
    sc = scenes.small_two_scale(nx=4, ny=4, mode=mode, split_x=split_x)
    got = []
    for cap in (last[0], last[0] + 1, last[1], last[1] + 1):
        sol = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
        got.append(sol.lanes())
        sol.close()
    assert got == [8, 4, 4, 1]
