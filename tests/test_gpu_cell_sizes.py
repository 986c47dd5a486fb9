"""The device's cell of a position (a corrected product with the reciprocal of
the cell size) is the division's for cell sizes of any mantissa: at and next to
powers of two, and drawn. Positions lie on and next to the cells' edges and past
the domain, where a quotient off by one unit would move a particle.
"""
from __future__ import annotations

import numpy as np
import pytest

from twoscalesplit_amd import MODE_PLAIN, Solver, config_init

pytestmark = pytest.mark.gpu


def _sizes():
    rng = np.random.default_rng(11)
    two = np.float32(2.0) ** np.arange(-7, 1, dtype=np.float32)
    near = [np.nextafter(t, np.float32(d)) for t in two[::2] for d in (0.0, 10.0)]
    drawn = (2.0 ** rng.uniform(-20.0, 20.0, 12)).astype(np.float32)
    return [float(v) for v in (*two[::3], *near, *drawn)]


@pytest.mark.parametrize("h", _sizes())
def test_cells(h):
    h = np.float32(h)
    dims = np.array([61, 47])
    end = (dims.astype(np.float32) * h).astype(np.float32)
    cfg = config_init(0.0, 0.0, float(end[0]), float(end[1]), float(h), float(h), 1.0, 1.0, 1.0,
                      0.1, 0.0, 1e-30)
    cfg.mode, cfg.cap_high = MODE_PLAIN, 0
    cfg.mass_low = cfg.mass_high = cfg.mass_boundary = 1.0
    dims = np.array(cfg.domain_dims)
    rng = np.random.default_rng(int(h.view(np.uint32)))
    n = 4000
    x = (rng.integers(-1, dims + 2, (n, 2)).astype(np.float32) * h).astype(np.float32)
    off = rng.integers(-2, 3, (n, 2))
    for k in (1, 2):
        x = np.where(off >= k, np.nextafter(x, np.float32(np.inf)), x)
        x = np.where(off <= -k, np.nextafter(x, np.float32(-np.inf)), x)
    x = x.astype(np.float32)
    t = (x + np.float32(0.0)) / h
    c = np.minimum(np.where(t >= 1.0, t, 0.0), (dims - 1).astype(np.float32)).astype(np.int64)
    want = np.bincount(c[:, 1] * dims[0] + c[:, 0], minlength=dims[0] * dims[1])
    bnd = np.array([[-10.0, -10.0]], np.float32) * h
    sol = Solver(cfg, x, n, bnd)
    try:
        sol.step(1)
        start, stop = sol.read("CELL_START_L"), sol.read("CELL_END_L")
        np.testing.assert_array_equal(np.where(start >= 0, stop - start, 0), want)
    finally:
        sol.close()
