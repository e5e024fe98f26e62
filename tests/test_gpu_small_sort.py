"""The one-launch update of a small scene's cell order: after every step the
order that step used equals std::stable_sort of the keys of the positions it
started from, at sizes around the update's tiles, from no particle changing
cell to all of them, through store reorders, rasters, state writes and graph
replays."""
from __future__ import annotations

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.solver import Solver
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def _check(gpu, desc, step, tag):
    pos = gpu.read_particles().position
    step()
    keys, ids, seq = gpu.read_sort()
    ref = pyoracle.keys(desc, pos[seq])
    order = pyoracle.stable_argsort(ref)
    moved = int((pyoracle.keys(desc, gpu.read_particles().position) != pyoracle.keys(desc, pos)).sum())
    assert np.array_equal(keys, ref[order]) and np.array_equal(ids, seq[order]), (tag, moved)
    return moved


@pytest.mark.parametrize("interp,transfer", [(N.QUADRATIC_BSPLINE, N.APIC), (N.LINEAR, N.PIC_FLIP),
                                             (N.CUBIC_BSPLINE, N.APIC)], ids=["quadratic", "linear", "cubic"])
@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 4097, 16384, 40000])
def test_order_is_the_stable_sort(n, interp, transfer):
    # (h = 1/32: x / h is exact, so that the oracle's keys are the device's also
    # at a cell's face.)  Random velocities of 0.3 cells per step (a quarter to all of the particles
    # of a step change cell), then a slow drift, then none
    sc = scenes.snow_cube(seed=n, n=n, res=32, transfer=transfer, interp=interp, dt=1e-4)
    gpu = Solver(sc.desc, sc.particles)
    r = np.random.default_rng(n)
    moves = []
    for speed in (0.3, 0.02, 0.0):
        st = gpu.read_particles()
        st.velocity[:] = r.normal(0, 1, (n, 3)) * speed / (32 * 1e-4) + np.array([speed, 0, 0]) / (32 * 1e-4)
        if st.B is not None:
            st.B[:] = 0.0
        gpu.write_particles(st)
        moves += [_check(gpu, sc.desc, lambda: gpu.step(1), (n, speed, k)) for k in range(4)]
    print(f"[update n={n} interp={interp}] particles that changed cell per step: {moves}", flush=True)


@pytest.mark.parametrize("transfer", [N.PIC_FLIP, N.APIC])
def test_order_through_other_calls(transfer):
    sc = scenes.snow_cube(seed=5, n=9000, res=32, transfer=transfer, dt=1e-4, velocity=(20.0, -7.0, 3.0))
    gpu = Solver(sc.desc, sc.particles)
    gpu.set_reorder_interval(3)
    one = lambda: gpu.step(1)  # noqa: E731
    for k in range(5):
        _check(gpu, sc.desc, one, ("reorder", k))
    gpu.density()  # sorts the current positions
    _check(gpu, sc.desc, one, "after a raster")
    _check(gpu, sc.desc, one, "after that")
    for k in range(7):  # with reorders between replays
        _check(gpu, sc.desc, lambda: gpu.step_graph(1), ("graph", k))
    _check(gpu, sc.desc, one, "eager after replays")
    st = gpu.read_particles()
    st.position[:, 2] += np.float32(0.05)
    gpu.write_particles(st)
    _check(gpu, sc.desc, lambda: gpu.step_graph(1), "graph after a state write")
    gpu.sort()
    _check(gpu, sc.desc, one, "after a sort")
    gpu.particlesToGrid()
    gpu.advectParticles(1e-4)
    _check(gpu, sc.desc, one, "after sub-steps")
    assert gpu.stats()["incremental_sorts"] == 0  # counted for scenes of 2^20 particles and up
