"""The cap on high particles where it cuts candidates: the first of them in
sorted order split, whatever part of a compaction tile (2048 entries) a scene's
segment begins and ends in; and the cut costs little.
"""
from __future__ import annotations

import time

import numpy as np
import pytest

from twoscalesplit_amd import MODE_REFERENCE, Batch, Solver, scenes

pytestmark = pytest.mark.gpu


def _scene(i, nx, ny, cap, split_x=-1.0):
    sc = scenes.small_two_scale(seed=i, nx=nx, ny=ny, nxd=2 * nx + 8, nyd=ny + 20,
                                mode=MODE_REFERENCE, split_x=split_x)
    sc.cfg.cap_high = min(cap, 4 * nx * ny)
    sc.cfg.time_step = 1e-5
    return sc


@pytest.mark.parametrize("allowed", [1, 255, 256, 257, 2047, 2048, 2049, 2900])
def test_first_candidates_split(allowed):
    # segments of 1, 255, 256, ... entries: the others begin anywhere in a tile
    sizes = [(1, 1), (15, 17), (50, 60), (16, 16), (53, 61), (7, 11), (64, 64), (50, 60)]
    scs = [_scene(i, nx, ny, 4 * allowed, 0.03 if i % 3 == 2 else -1.0)
           for i, (nx, ny) in enumerate(sizes)]
    print("[case]", allowed, flush=True)
    b = Batch(len(scs), sum(len(s.low_xy) for s in scs), sum(len(s.bnd_xy) for s in scs),
              sum(s.cells[0] for s in scs), sum(s.cells[1] for s in scs))
    try:
        ids = [b.add_scene(s.cfg, s.low_xy, len(s.low_xy), s.bnd_xy) for s in scs]
        for step in (1, 2):
            before = [b.read(i, "STATE_L") for i in ids]
            counts = [b.counts(i) for i in ids]
            b.step(1)
            for i, sc, st, c0 in zip(ids, scs, before, counts):
                c = b.counts(i)
                order = b.read(i, "SORTED_L", c)
                x = b.read(i, "POS_L", c)[:, 0]
                cand = order[(st[order] == 0) & (x[order] > np.float32(sc.cfg.split_x))]
                want = cand[:max(0, min(allowed, len(sc.low_xy)) - c0["n_groups"])]
                assert c["n_split"] == len(want)
                groups = b.read(i, "LIST_G", c)
                np.testing.assert_array_equal(groups[c0["n_groups"]:], want)
                assert c["n_high"] == 4 * len(groups) == len(b.read(i, "LIST_H", c))
    finally:
        b.close()


def test_a_binding_cap_costs_little():
    """90,000 low ids, half of them candidates under a cap of 200 splits: with an
    atomic per entry cut a step took 7.5 times what it takes without the cap."""
    us = {}
    for cap in (800, 360000):
        sc = _scene(1, 300, 300, cap, 150 / 160.0)
        sol = Solver(sc.cfg, sc.low_xy, len(sc.low_xy), sc.bnd_xy)
        try:
            sol.step(2)
            sol.step_graph(10)
            sol.synchronize()
            us[cap] = 1e9
            for _ in range(5):
                t = time.perf_counter()
                sol.step_graph(20)
                sol.synchronize()
                us[cap] = min(us[cap], (time.perf_counter() - t) / 20 * 1e6)
        finally:
            sol.close()
    print("[us]", us, flush=True)
    assert us[800] < 4.0 * us[360000]
