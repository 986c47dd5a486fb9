"""Blocks of the force sums with one lane per target: the walk closes a block
at every 16th iteration as long as each recorded candidate was a pair, and
counts from the first one that was none (a coincident particle, r = 0, or one
at the cutoff, r = h). Against the kernel with several lanes per target, which
counts every pair: the same bits, with none, few and many such candidates, in
scenes of one and two levels, and with more pairs than a block.
"""
from __future__ import annotations

import numpy as np
import pytest

from twoscalesplit_amd import MODE_PLAIN, MODE_REFERENCE, Solver, _native as N, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("twins", [0, 1, 7, 120])
@pytest.mark.parametrize("lattice", [False, True])
def test_blocks(two, twins, lattice):
    sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_REFERENCE if two else MODE_PLAIN,
                                split_x=0.05)
    n = len(sc.low_xy)
    if lattice:
        i = np.arange(n)
        sc.low_xy = ((np.stack([i % 24, i // 24], 1) + 0.5) / 160.0).astype(np.float32)
    rng = np.random.default_rng(twins)
    at = rng.permutation(n)
    sc.low_xy = sc.low_xy.copy()
    sc.low_xy[at[:twins]] = sc.low_xy[at[twins:2 * twins]]
    # closer: more pairs than two blocks
    sc.low_xy = (sc.low_xy * np.float32(0.75) + np.float32(0.01)).astype(np.float32)
    sc.cfg.time_step = 1e-6
    print("[case]", two, twins, lattice, flush=True)
    a = Solver(sc.cfg, sc.low_xy, 2 * n, sc.bnd_xy)
    b = Solver(sc.cfg, sc.low_xy, 2 * n, sc.bnd_xy)
    try:
        b.set_tuning(N.TssTuning.uniform())
        for steps in (1, 2, 4):
            a.step(steps)
            b.step_graph(steps)
            sa, sb = a.snapshot(), b.snapshot()
            assert sa.pop("counts") == sb.pop("counts")
            for f in sa:
                np.testing.assert_array_equal(sa[f], sb[f], err_msg=f)
    finally:
        a.close()
        b.close()
