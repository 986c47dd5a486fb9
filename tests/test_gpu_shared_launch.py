"""Both levels' neighbour sums in one launch (scenes of two levels, one lane per
target, the levels' launch shapes equal) against a launch per level (shapes
that differ): the same bits, from the first step (no high particle) on, with
counts around a block's, one scene and several, and past the capacity up to
which a launch is shared. A batch with a band-rule scene cuts the high level's
blocks to 262144 targets: with more, a scene is what it is alone.
"""
from __future__ import annotations

import numpy as np
import pytest

from twoscalesplit_amd import (MODE_BAND, MODE_PLAIN, MODE_REFERENCE, Batch, Solver,
                               _native as N, scenes)

pytestmark = pytest.mark.gpu


def _own(block_high):
    t = N.TssTuning.uniform(256, 16, 0, 0)
    t.block[1] = t.block[3] = block_high
    return t


@pytest.mark.parametrize("nx,ny", [(1, 1), (15, 17), (16, 16), (257, 1), (24, 30)])
@pytest.mark.parametrize("mode", [MODE_BAND, MODE_REFERENCE])
@pytest.mark.parametrize("cap", [60000, 262145])
def test_one_scene(nx, ny, mode, cap):
    sc = scenes.small_two_scale(nx=nx, ny=ny, nxd=max(48, nx + 8), mode=mode, split_x=0.05)
    print("[case]", nx, ny, mode, cap, flush=True)
    a = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    b = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    try:
        b.set_tuning(_own(128))
        for steps in (1, 1, 3):
            a.step_graph(steps)
            b.step(steps)
            sa, sb = a.snapshot(), b.snapshot()
            assert sa.pop("counts") == sb.pop("counts")
            for f in sa:
                np.testing.assert_array_equal(sa[f], sb[f], err_msg=f)
    finally:
        a.close()
        b.close()


def test_several_scenes():
    scs = [scenes.small_two_scale(nx=24, ny=30, mode=m, split_x=0.05)
           for m in (MODE_REFERENCE, MODE_PLAIN, MODE_BAND)]
    out = []
    for own in (False, True):
        b = Batch(3, 90000, sum(len(s.bnd_xy) for s in scs), sum(s.cells[0] for s in scs),
                  sum(s.cells[1] for s in scs))
        try:
            ids = [b.add_scene(s.cfg, s.low_xy, 30000, s.bnd_xy) for s in scs]
            if own:
                b.set_tuning(_own(512))
            b.step_graph(4)
            out.append([b.snapshot(i).copy() for i in ids])
        finally:
            b.close()
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)


def test_more_high_targets_than_blocks_of_a_band_batch():
    big = scenes.small_two_scale(nx=280, ny=250, nxd=300, nyd=260, mode=MODE_REFERENCE,
                                 split_x=-1.0)
    band = scenes.small_two_scale(nx=24, ny=30, mode=MODE_BAND)
    scs = (big, band)
    b = Batch(2, sum(len(s.low_xy) for s in scs), sum(len(s.bnd_xy) for s in scs),
              sum(s.cells[0] for s in scs), sum(s.cells[1] for s in scs))
    a = Solver(big.cfg, big.low_xy, len(big.low_xy), big.bnd_xy)
    try:
        ids = [b.add_scene(s.cfg, s.low_xy, len(s.low_xy), s.bnd_xy) for s in scs]
        for steps in (2, 3):
            a.step_graph(steps)
            b.step_graph(steps)
        assert a.counts()["n_high"] == 280000
        for f in ("POS_H", "VEL_H", "RHO_H", "POS_L", "VEL_L", "RHO_L"):
            np.testing.assert_array_equal(a.read(f), b.read(ids[0], f), err_msg=f)
    finally:
        a.close()
        b.close()
