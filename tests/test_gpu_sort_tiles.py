"""The cell order of a large scene at the edges of the sort's tiles (2,048
entries): a step's order equals std::stable_sort of the keys of the positions
it started from, whether the update made it (above 8,192 tiles their shifts
are scanned by a launch of their own) or, as the move list or a tile's bucket
overflowed, the full sort in one launch."""
from __future__ import annotations

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.batch import Batch
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


@pytest.mark.parametrize("n", [2**20, 2**20 + 1, 2**20 + 2047])
def test_full_sort_in_one_launch(n):
    # half a cell per step: far more moves than the list holds
    sc = scenes.snow_cube(seed=4, n=n, res=64, lo=0.25, hi=0.5, transfer=N.PIC_FLIP, dt=1e-4,
                          velocity=(0.5e4 / 64, 0.0, -0.1e4 / 64))
    gpu = Solver(sc.desc, sc.particles)
    gpu.set_reorder_interval(0)
    gpu.step(1)
    for k in range(2):
        pos = gpu.read_positions4()[:, :3]
        gpu.step(1)
        keys, ids, seq = gpu.read_sort()
        ref = pyoracle.keys(sc.desc, pos[seq])
        order = pyoracle.stable_argsort(ref)
        assert np.array_equal(keys, ref[order]) and np.array_equal(ids, seq[order]), (n, k)
    assert gpu.stats()["incremental_sorts"] == 0
    gpu.close()


@pytest.mark.parametrize("sizes", [(2048,), (2049,), (1000, 5000, 1)])
def test_full_sort_in_one_launch_of_a_small_batch(sizes):
    # fewer tiles than workgroups; a tile's bucket overflows, not the list
    b = Batch(N.QUADRATIC_BSPLINE, N.PIC_FLIP)
    scs = [scenes.snow_cube(seed=k, n=n, res=32, lo=0.25, hi=0.5, transfer=N.PIC_FLIP, dt=1e-4,
                            velocity=(0.5e4 / 32, 0.0, -0.1e4 / 32)) for k, n in enumerate(sizes)]
    solvers = [Solver(sc.desc, sc.particles) for sc in scs]
    for s in solvers:
        b.add(s)
    b.set_reorder_interval(0)
    seqs = []  # each member's store order, which the slots count in
    for s in solvers:
        s.sort()
        seqs.append(s.read_sort()[2])
    for k in range(3):
        pos = [s.read_particles().position[q] for s, q in zip(solvers, seqs)]
        b.step(1)
        keys, slots = b.read_sort()
        local = np.concatenate([pyoracle.keys(sc.desc, p).astype(np.int64) for sc, p in zip(scs, pos)])
        member = np.repeat(np.arange(len(sizes)), sizes)
        off = np.full(len(sizes), -1, np.int64)  # a member's key offset, from the sorted keys
        diff = keys.astype(np.int64) - local[slots]
        for j in range(len(sizes)):
            off[j] = diff[member[slots] == j][0]
        whole = local + off[member]
        order = np.lexsort((np.arange(whole.size), whole))
        assert np.array_equal(slots, order) and np.array_equal(keys, whole[order]), (sizes, k)
    assert b.info()["incremental_sorts"] == 0
    b.close()
    for s in solvers:
        s.close()
