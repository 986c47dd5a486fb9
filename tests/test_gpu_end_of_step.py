"""The next lists of a step: entries that a raw device pointer marked as
deleted leave the low list, in order and in any number around a compaction
tile (2048 entries), and a plain scene without such a pointer keeps its
list. The expected list is the step's sorted ids without them.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from twoscalesplit_amd import MODE_BAND, MODE_PLAIN, Solver, scenes

pytestmark = pytest.mark.gpu


def _to_device(ptr, arr):
    """A program's own copy into the solver's memory (hipMemcpy)."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    assert hip.hipMemcpy(ptr, arr.ctypes.data, arr.nbytes, 1) == 0


@pytest.mark.parametrize("mode", [MODE_PLAIN, MODE_BAND])
@pytest.mark.parametrize("nx,ny", [(1, 1), (45, 45), (64, 32), (2049, 1), (97, 83)])
def test_deleted_by_device_pointer_leave_the_list(mode, nx, ny):
    sc = scenes.small_two_scale(nx=nx, ny=ny, nxd=2 * nx + 8, nyd=ny + 40, mode=mode)
    print("[case]", mode, nx, ny, flush=True)
    sol = Solver(sc.cfg, sc.low_xy, sc.cap_low, sc.bnd_xy)
    try:
        sol.step(2)
        c = sol.counts()
        if mode == MODE_PLAIN:
            np.testing.assert_array_equal(sol.read("LIST_L", c), sol.read("SORTED_L", c))
        ptr = sol.device_ptr("STATE_L")
        state = sol.read("STATE_L", c)
        gone = np.flatnonzero((state == 0) & (np.arange(nx * ny) % 3 == 0))
        state[gone] = 2
        _to_device(ptr, state)
        sol.step(1)
        c = sol.counts()
        order = sol.read("SORTED_L", c)
        want = order[~np.isin(order, gone)]
        np.testing.assert_array_equal(sol.read("LIST_L", c), want)
        assert c["n_low"] == len(want) and c["n_low_last"] == len(order)
        sol.step_graph(3)
        assert sol.counts()["n_low_last"] == len(want)
    finally:
        sol.close()
