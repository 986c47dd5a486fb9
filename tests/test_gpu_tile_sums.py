"""The next lists of a step whose compaction tiles are summed in groups of 256
(capacities of more than 4096 tiles, 2048 entries each) are those of the same
scene in a capacity of fewer tiles: splits, and entries deleted through a device
pointer, in lists of one, a few and many groups of tiles.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from twoscalesplit_amd import MODE_BAND, MODE_REFERENCE, Solver, scenes

pytestmark = pytest.mark.gpu


def _delete(sol, gone):
    """States written by a program's own copy into the solver's memory."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    ptr = sol.device_ptr("STATE_L")
    state = sol.read("STATE_L")
    state[gone] = 2
    assert hip.hipMemcpy(ptr, state.ctypes.data, state.nbytes, 1) == 0


@pytest.mark.parametrize("nx,ny,mode", [
    (1, 1, MODE_REFERENCE), (64, 32, MODE_REFERENCE), (97, 83, MODE_BAND),
    (1024, 512, MODE_REFERENCE),      # low tiles: 256, a whole group
    (1025, 512, MODE_REFERENCE),
    (1500, 800, MODE_REFERENCE)])     # 3, 5 and 2 groups of tiles
def test_lists(nx, ny, mode):
    sc = scenes.small_two_scale(nx=nx, ny=ny, nxd=nx + 40, nyd=ny + 40, mode=mode,
                                split_x=0.5 * nx / 160.0)
    n = nx * ny
    print("[case]", nx, ny, mode, flush=True)
    out = []
    for cap in (n, 1500000):
        sol = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
        try:
            got = []
            for k in range(3):
                sol.step(1)
                c = sol.counts()
                got.append([c["n_low"], c["n_high"], c["n_groups"], c["n_split"]])
                got += [sol.read(f, c) for f in ("LIST_L", "LIST_H", "LIST_G")]
                if k == 0:
                    # active ones only: a parent's group keeps its children
                    state = sol.read("STATE_L", c)[:n]
                    _delete(sol, np.flatnonzero((state == 0) & (np.arange(n) % 3 == 0)))
            sol.step_graph(2)
            got.append(sol.read("LIST_L"))
            out.append(got)
        finally:
            sol.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    assert mode != MODE_REFERENCE or n == 1 or out[0][0][3] > 0.4 * n
