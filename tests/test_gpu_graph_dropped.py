"""A captured step that is dropped and captured again while its replays are
still queued: the calls do not wait in between, and the particles end where the
same steps run one by one put them."""
from __future__ import annotations

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.batch import Batch, Tune
from mpm_amd.solver import Solver

pytestmark = pytest.mark.gpu


def close_to(a, b):
    # the order of the grid's atomics differs from run to run: 60 steps of
    # 2^-24 each, amplified a little by the deformation
    x, y = a.position.astype(np.float64), b.position.astype(np.float64)
    assert np.abs(x - y).max() <= 1e-5, np.abs(x - y).max()


def test_scene():
    sc = scenes.snow_cube(seed=7, n=60_000, res=64, transfer=N.APIC, dt=1e-4, velocity=(1.0, -2.0, 0.5))
    a, b = Solver(sc.desc, sc.particles), Solver(sc.desc, sc.particles)
    for k in range(4):
        a.step_graph(15)  # returns before its replays have run
        a.set_particles_collision(k % 2 == 0)
        b.step(15)
        b.set_particles_collision(k % 2 == 0)
    assert a.stats()["graph_captures"] == 4
    close_to(a.read_particles(), b.read_particles())
    a.close()
    b.close()


def test_batch():
    sizes = (30_000, 5_000, 60_000)
    scs = [scenes.snow_cube(seed=k, n=n, res=64, transfer=N.APIC, dt=1e-4, velocity=(1.0, -2.0, 0.5))
           for k, n in enumerate(sizes)]
    runs = []
    for graph in (True, False):
        solvers = [Solver(sc.desc, sc.particles) for sc in scs]
        b = Batch(N.QUADRATIC_BSPLINE, N.APIC)
        for s in solvers:
            b.add(s)
        for item_max in (512, 128, 256, 512):
            b.set_tune(Tune(item_max=item_max, g2p_threads=128, workgroups=0, fuse_transfer=0))
            (b.step_graph if graph else b.step)(15)
        runs.append([s.read_particles() for s in solvers])
        b.close()
        for s in solvers:
            s.close()
    for x, y in zip(*runs):
        close_to(x, y)
