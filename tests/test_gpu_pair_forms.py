"""Pair sets (tss_pair_sets) are recorded by the form of the neighbour kernels
that a step takes: one, four or eight lanes per target. Each form's sets are
the oracle's, on targets that fit a group's LDS and that do not (crowded), at
the cutoff (an unjittered lattice), with promoted children and in scenes of one
level; and the library holds a recording instance of each form.
"""
from __future__ import annotations

import re

import numpy as np
import pytest
from parity import check_pairs

from oracle import binding as ob
from twoscalesplit_amd import MODE_BAND, MODE_PLAIN, MODE_REFERENCE, Solver, _native as N, scenes


def test_every_form_has_a_recording_instance():
    names = open(N.LIB_PATH, "rb").read()
    for kernel in (b"k_density_coop", b"k_force_coop"):
        lanes = {int(m) for m in re.findall(kernel + rb"ILi(\d)ELb1E", names)}
        assert lanes == {4, 8}, (kernel, lanes)


def _scene(kind):
    if kind == "plain":
        sc = scenes.small_two_scale(nx=23, ny=29, mode=MODE_PLAIN)
    elif kind == "band":
        sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_BAND)
        sc.cfg.promote_min_age, sc.cfg.promote_max_age = 2, 4
    else:
        sc = scenes.small_two_scale(nx=24, ny=30, mode=MODE_REFERENCE, split_x=0.05)
    if kind == "lattice":
        i = np.arange(24 * 30)
        sc.low_xy = ((np.stack([i % 24, i // 24], 1) + 0.5) / 160.0).astype(np.float32)
    if kind.startswith("crowd"):
        f = np.float32(float(kind[5:]) / 100.0)
        sc.low_xy = (sc.low_xy * f + np.float32(0.02)).astype(np.float32)
        sc.cfg.time_step = 1e-6
    return sc


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "band", "two", "lattice", "crowd70", "crowd30"])
@pytest.mark.parametrize("lanes", [1, 4, 8])
def test_pair_sets_of_each_form(kind, lanes):
    sc = _scene(kind)
    # the capacity picks the lanes
    cap = {8: 5000, 4: 16000, 1: 60000}[lanes]
    if sc.cfg.mode != MODE_REFERENCE and lanes == 4:
        cap = 48000
    print("[case]", kind, lanes, flush=True)
    sol = Solver(sc.cfg, sc.low_xy, cap, sc.bnd_xy)
    try:
        for steps in (0, 1, 5):
            sol.step(steps)
            o = ob.Scene(ob.params_from_config(sc.cfg), cap, sc.bnd_xy)
            o.load_snapshot(sol.snapshot())
            n, nh = check_pairs(sol, o, o.grid())
            assert n == sol.counts()["n_low"] and nh == sol.counts()["n_high"]
    finally:
        sol.close()
