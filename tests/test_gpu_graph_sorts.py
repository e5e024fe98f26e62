"""The sort of a captured step over a long run: the form of it that most steps
need is captured again in the middle of a call, and the updates go on
afterwards.  How often the update ran is read back without waiting, so the
calls below are short and waited for."""
from __future__ import annotations

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.solver import Solver
from oracle import pyoracle
from tests.test_gpu_batch_replay import check_step, make_batch

pytestmark = pytest.mark.gpu


def replay(gpu, steps, per_call=4):
    for _ in range(0, steps, per_call):
        gpu.step_graph(per_call)
        gpu.synchronize()
    return gpu.stats()


def check_order(gpu, desc, tag):
    """One more replay: its order is the stable sort of the positions before it."""
    pos = gpu.read_positions4()[:, :3]
    gpu.step_graph(1)
    keys, ids, seq = gpu.read_sort()
    ref = pyoracle.keys(desc, pos[seq])
    order = pyoracle.stable_argsort(ref)
    assert np.array_equal(keys, ref[order]) and np.array_equal(ids, seq[order]), tag


def test_capture_beside_a_reorder_keeps_the_update():
    sc = scenes.apic_slab(seed=7, nx=128, ny=64, nz=128, res=128, dt=5e-5, sigma_v=2.0)
    gpu = Solver(sc.desc, sc.particles)
    # a reorder before every replay: each sorts in full, so the full sort is
    # captured again pass by pass, in the same turn as a reorder
    gpu.set_reorder_interval(1)
    st = replay(gpu, 48)
    assert st["incremental_sorts"] == 0 and st["graph_captures"] == 2
    check_order(gpu, sc.desc, "full sorts")
    # none any more: the replays update, and the light form comes back
    gpu.set_reorder_interval(0)
    st = replay(gpu, 48)
    assert st["incremental_sorts"] >= 46 and st["graph_captures"] == 3, st
    check_order(gpu, sc.desc, "updates")
    gpu.close()


def test_batch_between_full_sorts_and_updates():
    # 0.4 cells per step: tiles of the order draw more than their buckets hold,
    # every replay sorts in full (captured again pass by pass); then at rest
    b, scs, solvers, seqs = make_batch((3000, 2500, 4000), velocity=(0.4e4 / 32, 0.0, -0.1e4 / 32))

    def run(steps):
        for _ in range(0, steps, 4):
            b.step_graph(4)
            b.synchronize()
        check_step(b, scs, solvers, seqs, lambda: b.step_graph(1), "replay")
        check_step(b, scs, solvers, seqs, lambda: b.step(1), "eager")
        return b.info()["incremental_sorts"]

    assert run(20) == 0
    for s in solvers:
        st = s.read_particles()
        st.velocity[:] = 0.0
        s.write_particles(st)
    assert run(40) >= 38
    b.close()
    for s in solvers:
        s.close()


@pytest.mark.parametrize("graph", [True, False], ids=["graph", "eager"])
@pytest.mark.parametrize("n,cells", [(16_384, 0.1), (16_384, 0.4), (100_000, 0.1), (100_000, 0.4), (200_000, 0.4),
                                     (1_000_000, 0.02), (1_000_000, 0.1)])
def test_small_scene_between_radix_sort_and_update(n, cells, graph):
    # the line: a fifth of the particles, or 20,000 and a 32nd (26,250 of
    # 200,000); then at rest
    radix = n * cells > min(n / 5, 20000 + n / 32)
    sc = scenes.snow_cube(seed=9, n=n, res=64, lo=0.25, hi=0.5, transfer=N.PIC_FLIP, dt=1e-4,
                          velocity=(cells * 1e4 / 64, 0.0, 0.0))
    gpu = Solver(sc.desc, sc.particles)
    step = gpu.step_graph if graph else gpu.step

    def run(steps):
        for _ in range(0, steps, 4):
            step(4)
            gpu.synchronize()
        for k in range(2):
            pos = gpu.read_positions4()[:, :3]
            step(1)
            keys, ids, seq = gpu.read_sort()
            ref = pyoracle.keys(sc.desc, pos[seq])
            order = pyoracle.stable_argsort(ref)
            assert np.array_equal(keys, ref[order]) and np.array_equal(ids, seq[order]), k
        return gpu.stats()["graph_captures"]

    captures = run(20)
    assert captures == (1 + radix if graph else 0)
    st = gpu.read_particles()
    st.velocity[:] = 0.0
    gpu.write_particles(st)
    assert run(24) == (captures + radix if graph else 0)
    gpu.close()


@pytest.mark.parametrize("interval", [3, 5, 10])
def test_captures_settle(interval):
    # a reorder, and with it a full sort, every few replays: at 2/3 or 4/5
    # updates the full sort is launched pass by pass, captured so once; at 9/10
    # it stays the light one
    sc = scenes.apic_slab(seed=7, nx=128, ny=64, nz=128, res=128, dt=5e-5, sigma_v=2.0)
    gpu = Solver(sc.desc, sc.particles)
    gpu.set_reorder_interval(interval)
    st = replay(gpu, 120)
    assert st["graph_captures"] == (1 if interval == 10 else 2), st
    assert st["incremental_sorts"] >= 120 - 120 // interval - 2
    gpu.close()


def test_moves_that_overflow_and_back():
    # 0.3 cells per step of 1.1M particles: the list, then the buckets, overflow
    # and every replay sorts in full; at rest the updates come back
    sc = scenes.snow_cube(seed=8, n=1_100_000, res=64, lo=0.25, hi=0.5, transfer=N.PIC_FLIP, dt=1e-4,
                          velocity=(0.3e4 / 64, 0.0, 0.0))
    gpu = Solver(sc.desc, sc.particles)
    gpu.set_reorder_interval(0)
    st = replay(gpu, 20)
    assert st["incremental_sorts"] == 0 and st["graph_captures"] == 2, st
    check_order(gpu, sc.desc, "full sorts")
    state = gpu.read_particles()
    state.velocity[:] = 0.0
    gpu.write_particles(state)
    st = replay(gpu, 48)
    assert st["incremental_sorts"] >= 46 and st["graph_captures"] == 3, st
    check_order(gpu, sc.desc, "updates")
    gpu.close()
