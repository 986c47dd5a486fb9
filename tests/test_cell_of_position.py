"""The cell of a position: the device takes the quotient by the cell size as a
product with the rounded reciprocal and two exact residual corrections. It has
to be the division's cell for every input: the arithmetic on the CPU (near
cell edges, any bits), and the device's cells themselves, also for cells of
extreme size, which keep the division.
"""
from __future__ import annotations

import ctypes
import ctypes.util

import numpy as np
import pytest

from twoscalesplit_amd import MODE_PLAIN, Solver, config_init, scenes


def _cell(t, dim):
    with np.errstate(invalid="ignore"):
        t = np.where(t >= 1.0, t, 0.0)
        return np.minimum(t, dim - 1).astype(np.int64)


def test_corrected_product_is_the_quotient():
    f = ctypes.CDLL(ctypes.util.find_library("m")).fmaf
    f.restype, f.argtypes = ctypes.c_float, [ctypes.c_float] * 3
    fma = np.frompyfunc(f, 3, 1)
    rng = np.random.default_rng(3)
    n = 60000
    c = rng.integers(0x21800000, 0x5D800000, n).astype(np.uint32).view(np.float32)
    edge = (c * rng.integers(0, 100000, n)).astype(np.float32)
    edge = (edge.view(np.uint32) + rng.integers(-3, 4, n).astype(np.uint32)).view(np.float32)
    any_bits = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32).view(np.float32)
    a = np.where(rng.random(n) < 0.7, edge, any_bits)
    a[:4] = np.inf, -np.inf, np.nan, 0.0
    with np.errstate(all="ignore"):
        inv = np.float32(1.0) / c
        q = a * inv
        t = q
        for _ in range(2):
            r = fma(-c, t, a).astype(np.float32)
            t = fma(r, inv, t).astype(np.float32)
        t = np.where(q < np.float32(1e9), t, q)
        ref = a / c
    dim = rng.integers(1, 200000, n)
    np.testing.assert_array_equal(_cell(t, dim), _cell(ref, dim))


@pytest.mark.gpu
@pytest.mark.parametrize("exponent", [0, -20, 40, -58, 66])
def test_cells_of_particles(exponent):
    """Cell sizes 0.02 * 2^exponent; the last two take the division."""
    s = np.float32(2.0) ** exponent
    base = scenes.small_two_scale(nx=24, ny=30, mode=MODE_PLAIN)
    b = base.cfg
    h, H = np.float32(b.effective_radius) * s, np.float32(b.effective_radius_high) * s
    end = [float(np.float32(v) * s) for v in b.domain_end]
    cfg = config_init(0.0, 0.0, *end, float(h), float(H), 1.0, 1.0, 1.0, 0.1, 0.0, 1e-30)
    cfg.mode, cfg.cap_high = MODE_PLAIN, 0
    cfg.mass_low = cfg.mass_high = cfg.mass_boundary = 1.0
    rng = np.random.default_rng(exponent + 100)
    n = 720
    dims = np.array(cfg.domain_dims)
    # on and next to the cells' edges, and past the domain on both sides
    x = (rng.integers(-1, dims + 2, (n, 2)) * h).astype(np.float32)
    x = np.where(rng.random((n, 2)) < 0.3, np.nextafter(x, np.float32(np.inf)), x)
    x = np.where(rng.random((n, 2)) < 0.3, np.nextafter(x, np.float32(-np.inf)), x)
    x = x.astype(np.float32)
    t = (x + np.float32(0.0)) / h
    c = _cell(t, dims)
    want = np.bincount(c[:, 1] * dims[0] + c[:, 0], minlength=dims[0] * dims[1])
    print("[case]", exponent, flush=True)
    sol = Solver(cfg, x, n, (base.bnd_xy * s).astype(np.float32))
    try:
        sol.step(1)
        start, end = sol.read("CELL_START_L"), sol.read("CELL_END_L")
        np.testing.assert_array_equal(np.where(start >= 0, end - start, 0), want)
    finally:
        sol.close()
