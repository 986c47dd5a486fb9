"""Supports of five and more particle spacings: a target's rows need more than
the eight words of a record. The density's sums take any number of words (one
lane per target), as those with several lanes per target and their scans do:
the same bits, in one level and two, and a step of them costs what its pairs do.
"""
from __future__ import annotations

import math
import time

import numpy as np
import pytest

from twoscalesplit_amd import MODE_BAND, MODE_PLAIN, MODE_REFERENCE, Solver, config_init, scenes
from twoscalesplit_amd import _native as N

pytestmark = pytest.mark.gpu


def _scene(nx, ny, support, mode):
    dx = 1.0 / 160.0
    low, bnd = scenes.generate(5, 1, nx, ny, dx, 2 * nx + 20, ny + 40)
    h = np.float32(support * dx)
    H = h if mode == MODE_PLAIN else np.float32(0.5) * h
    c0 = 10.0 * math.sqrt(2.0 * scenes.G * ny * dx)
    cfg = config_init(0.0, 0.0, (2 * nx + 20) * dx, (ny + 40) * dx, float(h), float(H),
                      scenes.RHO0, scenes.RHO0 * c0 * c0 / 7.0, c0, 0.05, 0.0, 1e-6)
    m = np.float32(scenes.RHO0 * dx * dx)
    cfg.mass_low = cfg.mass_boundary = float(m)
    cfg.mass_high = float(m) if mode == MODE_PLAIN else float(m / np.float32(4))
    cfg.mode, cfg.split_x = mode, 0.5 * nx * dx
    cfg.promote_min_age, cfg.promote_max_age = 2, 4
    return cfg, low, bnd


# 4.8 spacings: about as many targets with a record as without
@pytest.mark.parametrize("support", [4.8, 5.0, 6.0, 9.0, 14.0])
@pytest.mark.parametrize("mode", [MODE_PLAIN, MODE_REFERENCE, MODE_BAND])
def test_same_bits(support, mode):
    cfg, low, bnd = _scene(33, 47, support, mode)
    print("[case]", support, mode, flush=True)
    a = Solver(cfg, low, 5000, bnd)
    b = Solver(cfg, low, 5000, bnd)
    try:
        assert a.lanes() == 8
        b.set_tuning(N.TssTuning.uniform(128, 8, 1, 0))
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


def test_cost_of_a_wide_support():
    """At eight spacings a step has four times the pairs it has at four, and took
    5.9 times as long with a second scan, 4.0 times without."""
    us = {}
    for support in (4.0, 8.0):
        cfg, low, bnd = _scene(600, 500, support, MODE_PLAIN)
        sol = Solver(cfg, low, len(low), bnd)
        try:
            sol.step(2)
            sol.step_graph(10)
            sol.synchronize()
            us[support] = 1e9
            for _ in range(5):
                t = time.perf_counter()
                sol.step_graph(10)
                sol.synchronize()
                us[support] = min(us[support], (time.perf_counter() - t) / 10 * 1e6)
        finally:
            sol.close()
    print("[us]", us, flush=True)
    assert us[8.0] < 5.0 * us[4.0]
