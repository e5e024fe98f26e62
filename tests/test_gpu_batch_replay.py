"""A batch's captured step between eager ones: the order that a replay used is
the one that is read back, whichever form of the sort the eager step before it
took (the forms end in different buffers where their pass counts differ)."""
from __future__ import annotations

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.batch import Batch
from mpm_amd.solver import Solver
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def make_batch(sizes, velocity=(20.0, -7.0, 3.0), transfer=N.PIC_FLIP):
    scs = [scenes.snow_cube(seed=k, n=n, res=32, transfer=transfer, dt=1e-4, velocity=velocity)
           for k, n in enumerate(sizes)]
    solvers = [Solver(sc.desc, sc.particles) for sc in scs]
    b = Batch(N.QUADRATIC_BSPLINE, transfer)
    for s in solvers:
        b.add(s)
    b.set_reorder_interval(0)
    seqs = []  # each member's store order, which the slots count in
    for s in solvers:
        s.sort()
        seqs.append(s.read_sort()[2])
    return b, scs, solvers, seqs


def check_step(b, scs, solvers, seqs, step, tag):
    """The order of the step equals the stable sort of the positions before it."""
    pos = [s.read_particles().position[q] for s, q in zip(solvers, seqs)]
    step()
    keys, slots = b.read_sort()
    local = np.concatenate([pyoracle.keys(sc.desc, p).astype(np.int64) for sc, p in zip(scs, pos)])
    spans = [64 * (sc.desc.resolution[0] // 4 + 1) ** 3 + 64 for sc in scs]
    whole = local + np.repeat(np.concatenate([[0], np.cumsum(spans)[:-1]]), [len(p) for p in pos])
    order = np.lexsort((np.arange(whole.size), whole))
    assert np.array_equal(slots, order) and np.array_equal(keys, whole[order]), tag


def test_replay_after_an_eager_full_sort():
    # 18 key bits below 2^20 keys: the full sort takes two passes launched one
    # by one (9-bit digits) and three in one launch (8 bits)
    b, scs, solvers, seqs = make_batch((3000, 2500, 4000))
    assert b.info()["key_bits"] == 18
    for k in range(3):
        check_step(b, scs, solvers, seqs, lambda: b.step_graph(1), ("replay", k))
    solvers[1].advectParticles(1e-4)  # the keys are made anew: the next step sorts in full
    check_step(b, scs, solvers, seqs, lambda: b.step(1), "eager")
    for k in range(3):
        check_step(b, scs, solvers, seqs, lambda: b.step_graph(1), ("replay after it", k))
    b.close()
    for s in solvers:
        s.close()
