"""A batch of plain scenes launches nothing for high particles and copies its
lists, until the host gives it some or hands out a device pointer. Each such
change comes after steps were captured in a graph, and the scene then steps as
one whose rule has two levels (and splits nothing) from the start.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from twoscalesplit_amd import MODE_PLAIN, MODE_REFERENCE, Batch, Solver, scenes

pytestmark = pytest.mark.gpu

FIELDS = ("POS_L", "VEL_L", "ACC_L", "RHO_L", "P_L", "STATE_L", "AGE_L", "POS_H", "VEL_H",
          "ACC_H", "RHO_H", "P_H", "STATE_H", "LIST_L", "LIST_H", "LIST_G", "DT")


def _scene(mode, split_x=100.0):
    sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_REFERENCE, split_x=split_x)
    sc.cfg.mode = mode
    return sc


def _two_levels(cap):
    """A state with children (of the particles past x = 0.07)."""
    sc = _scene(MODE_REFERENCE, 0.07)
    with Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy) as s:
        s.step(3)
        snap = s.snapshot()
    assert snap["counts"]["n_high"] > 500
    return snap


def _same(a, b):
    for f in FIELDS:
        np.testing.assert_array_equal(a(f), b(f), err_msg=f)


# eight and four lanes per target and one, the levels in one launch and in two
@pytest.mark.parametrize("cap", [720, 30000, 60000, 262145])
@pytest.mark.parametrize("warm", [0, 4])
def test_children_from_the_host(cap, warm):
    snap = _two_levels(cap)
    plain, two = _scene(MODE_PLAIN), _scene(MODE_REFERENCE)
    print("[case]", cap, warm, flush=True)
    a = Solver(plain.cfg, plain.low_xy, cap, plain.bnd_xy)
    b = Solver(two.cfg, two.low_xy, cap, two.bnd_xy)
    try:
        for s in (a, b):
            s.step_graph(warm)
            s.restore(snap)
        for n in (1, 4, 2):
            for s in (a, b):
                s.step_graph(n)
            assert a.counts()["n_high"] == b.counts()["n_high"] > 500
            _same(a.read, b.read)
        # and back to one level: the lists alone
        for s in (a, b):
            low = s.read("STATE_L")
            low[:] = 0
            s.write("STATE_L", low)
            s.set_counts(s.counts()["n_low"], 0, 0)
            s.step_graph(4)
        assert a.counts()["n_high"] == 0
        _same(a.read, b.read)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("scenes_first", [0, 1])
def test_snapshot_with_children_into_a_plain_batch(scenes_first):
    snap = _two_levels(720)
    sc = _scene(MODE_PLAIN)
    a = Solver(sc.cfg, sc.low_xy, 720, sc.bnd_xy)
    a.restore(snap)
    a.step(1)
    saved = a.save_state()
    b = Batch(2, 1440, 2 * len(sc.bnd_xy), 2 * sc.cells[0], 2 * sc.cells[1])
    alone = Solver(sc.cfg, sc.low_xy, 720, sc.bnd_xy)
    try:
        if scenes_first:
            one = b.add_scene(sc.cfg, sc.low_xy, 720, sc.bnd_xy)
            b.step_graph(4)
        two = b.restore(saved)
        b.step_graph(5)
        a.step(5)
        _same(a.read, lambda f: b.read(two, f))
        if scenes_first:
            alone.step(9)
            _same(alone.read, lambda f: b.read(one, f))
    finally:
        a.close()
        b.close()
        alone.close()


@pytest.mark.parametrize("rule_gone", [False, True])
def test_last_two_level_scene_leaves(rule_gone):
    """The plain scene that stays steps as it does alone."""
    sc, other = _scene(MODE_PLAIN), _scene(MODE_REFERENCE, 0.07)
    b = Batch(2, 1440, 2 * len(sc.bnd_xy), 2 * sc.cells[0], 2 * sc.cells[1])
    a = Solver(sc.cfg, sc.low_xy, 720, sc.bnd_xy)
    try:
        gone = b.add_scene(other.cfg, other.low_xy, 720, other.bnd_xy)
        stays = b.add_scene(sc.cfg, sc.low_xy, 720, sc.bnd_xy)
        b.step_graph(4)
        assert b.counts(gone)["n_high"] > 0
        if rule_gone:
            b.remove_scene(gone)
        b.step_graph(5)
        a.step(9)
        _same(a.read, lambda f: b.read(stays, f))
        if rule_gone:
            again = b.add_scene(other.cfg, other.low_xy, 720, other.bnd_xy)
            b.step_graph(4)
            a.step(4)
            _same(a.read, lambda f: b.read(stays, f))
            assert b.counts(again)["n_high"] > 0
    finally:
        a.close()
        b.close()


def test_device_pointer_after_capture():
    """Entries deleted through a pointer handed out after steps were captured."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    sc = _scene(MODE_PLAIN)
    s = Solver(sc.cfg, sc.low_xy, 720, sc.bnd_xy)
    try:
        s.step_graph(4)
        ptr = s.device_ptr("STATE_L")
        for k, gone in enumerate((np.arange(0, 720, 7), np.arange(1, 720, 5))):
            state = s.read("STATE_L")
            state[gone] = 2
            assert hip.hipMemcpy(ptr, state.ctypes.data, state.nbytes, 1) == 0
            s.step_graph(2)
            low = s.read("LIST_L")
            assert not np.isin(gone, low).any()
            assert len(low) == np.count_nonzero(state != 2) == s.counts()["n_low"]
    finally:
        s.close()
