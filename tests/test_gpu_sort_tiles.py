"""The update of a large scene's cell order at the edges of its tiles (2,048
entries; above 8,192 tiles their shifts are scanned by a launch of their
own): the order of a step equals std::stable_sort of the keys of the
positions it started from, and the update made it."""
from __future__ import annotations

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.solver import Solver
from oracle import pyoracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,res", [(2**20, 64), (2**20 + 1, 64), (2**20 + 2047, 64), (8192 * 2048 + 1, 128)])
def test_order_is_the_stable_sort(n, res):
    # h is a power of two: the oracle's keys are the device's also at a cell's
    # face.  About a twentieth of the particles change cell in a step, the
    # last ones of the order among them (they drift up).
    sc = scenes.snow_cube(seed=3, n=n, res=res, lo=0.25, hi=0.75, transfer=N.PIC_FLIP, dt=1e-4,
                          velocity=(0.02 * 1e4 / res, 0.01 * 1e4 / res, 0.02 * 1e4 / res))
    gpu = Solver(sc.desc, sc.particles)
    gpu.set_reorder_interval(0)
    gpu.step(1)
    for k in range(2 if n < 2**21 else 1):
        pos = gpu.read_positions4()[:, :3]
        gpu.step(1)
        keys, ids, seq = gpu.read_sort()
        ref = pyoracle.keys(sc.desc, pos[seq])
        order = pyoracle.stable_argsort(ref)
        assert np.array_equal(keys, ref[order]) and np.array_equal(ids, seq[order]), (n, k)
        assert gpu.stats()["incremental_sorts"] == k + 1
    moved = int((pyoracle.keys(sc.desc, gpu.read_positions4()[:, :3]) != pyoracle.keys(sc.desc, pos)).sum())
    print(f"[update n={n}] particles that changed cell in the last step: {moved}", flush=True)
    assert moved > n // 100
    gpu.close()
