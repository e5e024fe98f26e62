"""A batch of many very small scenes: its health pass and its step do not take
a scene after the other (a workgroup of either spans hundreds of them)."""
from __future__ import annotations

import time

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.batch import Batch
from mpm_amd.solver import Solver

pytestmark = pytest.mark.gpu


def median_us(fn, times=15):
    t = []
    for _ in range(times):
        t0 = time.perf_counter()
        fn()
        t.append((time.perf_counter() - t0) * 1e6)
    return float(np.median(t))


def make(sizes, res=8):
    solvers = []
    for k, n in enumerate(sizes):
        sc = scenes.snow_cube(seed=k, n=max(n, 1), res=res, transfer=N.APIC)
        none = np.zeros((0, 3), np.float32)
        solvers.append(Solver(sc.desc, sc.particles if n else scenes.snow_particles(none, none, 1e-4)))
    b = Batch(N.QUADRATIC_BSPLINE, N.APIC)
    for s in solvers:
        b.add(s)
    return b, solvers


def close(b, solvers):
    b.close()
    for s in solvers:
        s.close()


def test_health_of_scenes_of_one_particle():
    # 256 scenes: the same reading, and the same host work per scene, for one
    # particle each (one workgroup has them all) as for 256 each (one apiece)
    one, big = make([1] * 256), make([256] * 256)
    t = [median_us(x[0].health) for x in (one, big)]
    print(f"[health] 256 scenes of 1 particle {t[0]:.0f} us, of 256 particles {t[1]:.0f} us", flush=True)
    assert t[0] < 1.5 * t[1] + 20
    for x in (one, big):
        close(*x)


@pytest.mark.parametrize("sizes", [(1,) * 70, (3, 0, 1, 250, 2, 2, 0, 64, 1, 1, 1, 300, 1, 1), (255, 1, 1, 1, 1, 255, 2)],
                         ids=["70", "14", "7"])
def test_health_of_mixed_waves(sizes):
    b, solvers = make(sizes)
    r = np.random.default_rng(1)
    want = []
    for i, (n, s) in enumerate(zip(sizes, solvers)):
        st = s.read_particles()
        st.velocity[:] = r.normal(0, 1, (n, 3)).astype(np.float32)
        off = r.choice(n, n // 3, replace=False) if n else []
        if n:
            st.position[off, i % 3] = 3.0
            st.velocity[0, 1] = np.inf if i % 3 == 0 else st.velocity[0, 1]
            s.write_particles(st)
        v = st.velocity.astype(np.float64)
        want.append((np.sqrt((v * v).sum(1).max()) if n else 0.0, int(n > 0 and i % 3 == 0), len(off)))
    for got, (speed, bad, off) in zip(b.health(), want):
        assert (got["nonfinite"], got["escaped"]) == (bad, off)
        # three roundings of the square, one of the root
        assert got["max_speed"] == speed or abs(got["max_speed"] - speed) <= 2.0**-21 * speed
    close(b, solvers)


def test_step_of_scenes_of_one_particle():
    # 900 scenes in one workgroup's run of keys, against 60 particles each:
    # fewer particles are not the longer step, and the scenes are the right ones
    one, more = make([1] * 900), make([60] * 900)
    t = []
    for b, _ in (one, more):
        def steps():
            b.step(20)
            b.synchronize()
        steps()
        t.append(median_us(steps) / 20)
    print(f"[step] 900 scenes of 1 particle {t[0]:.0f} us, of 60 particles {t[1]:.0f} us", flush=True)
    assert t[0] < t[1]
    for k in (0, 1, 63, 64, 450, 899):
        alone = Solver(scenes.snow_cube(seed=k, n=1, res=8, transfer=N.APIC).desc,
                       scenes.snow_cube(seed=k, n=1, res=8, transfer=N.APIC).particles)
        alone.step(20 * 16)
        x, y = one[1][k].read_particles(), alone.read_particles()
        # one particle falls freely: 320 steps of a few 2^-24 each
        assert np.abs(x.position.astype(np.float64) - y.position).max() <= 320 * 4 * 2.0**-24
        assert np.abs(x.velocity.astype(np.float64) - y.velocity).max() <= 320 * 4 * 2.0**-24
        alone.close()
    for x in (one, more):
        close(*x)
