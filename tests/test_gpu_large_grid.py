"""A few particles in a large, mostly empty grid: its clear reads a flag per
storage block and is a small part of the step."""
from __future__ import annotations

import time

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.solver import Solver

pytestmark = pytest.mark.gpu


def step_us(n, res, dt, transfer=N.PIC_FLIP):
    side = (n / 8) ** (1 / 3) / res  # 8 particles per cell
    sc = scenes.snow_cube(seed=1, n=n, res=res, lo=0.5 - side / 2, hi=0.5 + side / 2, transfer=transfer, dt=dt)
    s = Solver(sc.desc, sc.particles)
    s.step(3)
    s.synchronize()
    t = []
    for _ in range(9):
        t0 = time.perf_counter()
        s.step(20)
        s.synchronize()
        t.append((time.perf_counter() - t0) / 20e-6)
    st = s.stats()
    s.close()
    return float(np.median(t)), st


def test_clear_of_a_mostly_empty_grid():
    # 768^3: 7.1M storage blocks (18 GB), of which some hundreds are touched
    small, a = step_us(16384, 64, 1e-5)
    large, b = step_us(16384, 768, 1e-5)
    print(f"[large grid] step {small:.0f} us in 64^3, {large:.0f} us in 768^3", flush=True)
    assert large < 1.7 * small
    # every step's nodes were counted and cleared: as many per step in both, up
    # to where the body lies in the cells
    n = a["active_nodes_sum"] / a["steps"], b["active_nodes_sum"] / b["steps"]
    assert a["steps"] == b["steps"] == 183 and abs(n[0] / n[1] - 1) < 0.1


def test_fused_transfer_in_a_mostly_empty_grid():
    # APIC: two grids, cleared in turn beside the sort
    _, a = step_us(16384, 64, 1e-5, N.APIC)
    _, b = step_us(16384, 768, 1e-5, N.APIC)
    n = a["active_nodes_sum"] / a["steps"], b["active_nodes_sum"] / b["steps"]
    assert a["steps"] == b["steps"] == 183 and abs(n[0] / n[1] - 1) < 0.1
    assert a["escaped"] == b["escaped"] == 0
