"""The cut grid of the high level (batches with a band-rule scene): a band wide
enough to list more high targets than the grid holds loops over them, and beside
a reference-rule scene that lists as many the grid is whole. Either way a scene
is what it is alone, or what the oracle says.
"""
from __future__ import annotations

import numpy as np
import pytest
from parity import check_step

from twoscalesplit_amd import MODE_BAND, MODE_REFERENCE, Batch, Solver, scenes

pytestmark = pytest.mark.gpu


def test_wide_band_loops():
    sc = scenes.small_two_scale(nx=280, ny=250, nxd=600, nyd=300, mode=MODE_BAND)
    sc.cfg.band_radius = sc.cfg.merge_radius = 100 * sc.cfg.effective_radius
    sol = Solver(sc.cfg, sc.low_xy, len(sc.low_xy), sc.bnd_xy)
    try:
        sol.step(1)
        assert sol.counts()["n_high"] == 280000
        check_step(sol, sc.cfg, sc.bnd_xy, pairs=False)
    finally:
        sol.close()


def _batch(scs):
    return Batch(len(scs), sum(len(s.low_xy) for s in scs), sum(len(s.bnd_xy) for s in scs),
                 sum(s.cells[0] for s in scs), sum(s.cells[1] for s in scs))


# 4 * nx * ny around 262144, and below and above the low ids of a shared force
@pytest.mark.parametrize("nx,ny", [(256, 256), (257, 256), (560, 470)])
def test_beside_a_large_scene(nx, ny):
    big = scenes.small_two_scale(nx=nx, ny=ny, nxd=nx + 20, nyd=ny + 20, mode=MODE_REFERENCE,
                                 split_x=-1.0)
    band = scenes.small_two_scale(nx=24, ny=30, mode=MODE_BAND)
    print("[case]", nx, ny, flush=True)
    alone = [Solver(s.cfg, s.low_xy, len(s.low_xy), s.bnd_xy) for s in (big, band)]
    b = _batch((big, band))
    try:
        ids = [b.add_scene(s.cfg, s.low_xy, len(s.low_xy), s.bnd_xy) for s in (big, band)]
        b.step_graph(3)
        for i, a in zip(ids, alone):
            a.step(3)
            for f in ("POS_H", "VEL_H", "RHO_H", "POS_L", "VEL_L", "RHO_L", "LIST_H"):
                np.testing.assert_array_equal(a.read(f), b.read(i, f), err_msg=f)
    finally:
        b.close()
        for a in alone:
            a.close()
