"""Neighbour sums with several lanes per target (small batches) against one
lane per target (launch shapes set by the caller): the same bits, at target
counts around a block's (32 and 64), for targets that do not fit the group's
LDS (crowded: more pairs, words or rows than it holds), for pairs at the
cutoff (an unjittered lattice) and for every kernel form. The capacity picks
the lanes: up to 16384 expected targets eight, up to 49152 four.
"""
from __future__ import annotations

import numpy as np
import pytest

from twoscalesplit_amd import (MODE_BAND, MODE_PLAIN, MODE_REFERENCE, Solver,
                               _native as N, scenes)

pytestmark = pytest.mark.gpu


def _scene(kind):
    if kind[1:].isdigit():
        n = int(kind[1:])
        sc = scenes.small_two_scale(nx=n, ny=1, nxd=2 * n + 8, nyd=12,
                                    mode=MODE_PLAIN)
    elif kind == "band":
        sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_BAND)
        sc.cfg.promote_min_age, sc.cfg.promote_max_age = 2, 4
    else:
        ratio = {"wide": 0.6, "narrow": 0.3}.get(kind, 0.5)
        sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_REFERENCE,
                                    split_x=0.05, h_ratio=ratio)
    if kind == "tension":
        sc.cfg.tension_coefficient = 0.08
    if kind == "lattice":
        i = np.arange(24 * 30)
        sc.low_xy = ((np.stack([i % 24, i // 24], 1) + 0.5) / 160.0).astype(np.float32)
    if kind.startswith("crowd"):
        f = np.float32(float(kind[5:]) / 100.0)
        sc.low_xy = (sc.low_xy * f + np.float32(0.02)).astype(np.float32)
        sc.cfg.time_step = 1e-6
    return sc


@pytest.mark.parametrize("kind", ["n1", "n2", "n31", "n32", "n33", "n63", "n64", "n65",
                                  "band", "two", "wide", "narrow", "tension", "lattice",
                                  "crowd70", "crowd50", "crowd30"])
@pytest.mark.parametrize("expected", [16384, 49152])
def test_lanes_per_target_do_not_change_results(kind, expected):
    sc = _scene(kind)
    cap = expected // (3 if sc.cfg.mode == MODE_REFERENCE else 1)
    print("[case]", kind, expected, flush=True)
    a = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    b = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    try:
        b.set_tuning(N.TssTuning.uniform())
        for steps in (1, 1, 4, 6):
            a.step(steps)
            b.step_graph(steps)
            sa, sb = a.snapshot(), b.snapshot()
            assert sa.pop("counts") == sb.pop("counts")
            for f in sa:
                np.testing.assert_array_equal(sa[f], sb[f], err_msg=f)
    finally:
        a.close()
        b.close()
