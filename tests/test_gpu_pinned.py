"""What a scene's and a batch's sorts leave for the host lies in pinned memory
that outlives them: freeing a scene or a batch does not wait for the work that
other streams have queued."""
from __future__ import annotations

import time

import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.batch import Batch
from mpm_amd.solver import Solver, release_cache

pytestmark = pytest.mark.gpu


def test_destroy_does_not_wait_for_other_streams():
    slab = scenes.apic_slab(seed=2)  # 8.4M particles: 100 steps are ~0.13 s of queued work
    big = Solver(slab.desc, slab.particles)
    big.step(2)
    big.synchronize()
    mid = scenes.snow_cube(seed=5, n=150_000, res=64)
    one = Solver(mid.desc, mid.particles)
    one.step(10)
    one.synchronize()
    member = Solver(mid.desc, mid.particles)
    batch = Batch(N.QUADRATIC_BSPLINE, N.PIC_FLIP)
    batch.add(member)
    batch.step(10)
    batch.synchronize()
    t0 = time.perf_counter()
    big.step(100)
    t1 = time.perf_counter()
    one.close()
    batch.close()
    member.close()
    t2 = time.perf_counter()
    big.synchronize()
    t3 = time.perf_counter()
    print(f"[pinned] enqueue {1e3 * (t1 - t0):.1f} ms, destroy {1e3 * (t2 - t1):.1f} ms, "
          f"queued work left afterwards {1e3 * (t3 - t2):.1f} ms", flush=True)
    assert t3 - t2 > 0.02 and t2 - t1 < t3 - t1, (t1 - t0, t2 - t1, t3 - t2)
    big.close()


def test_words_of_many_scenes_and_after_a_release():
    # more scenes than a block has words, freed, given back, made again
    sc = scenes.snow_cube(seed=6, n=2**17, res=32, lo=0.25, hi=0.75)
    for _ in range(2):
        many = [Solver(sc.desc, sc.particles) for _ in range(66)]
        for s in many:
            s.step(9)  # writes its word
        release_cache()  # words in use stay
        for s in many:
            s.step(8)
        for s in many:
            assert s.stats()["steps"] == 17 and s.stats()["escaped"] == 0
            s.close()
        release_cache()
