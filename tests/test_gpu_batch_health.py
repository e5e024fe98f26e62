"""The health pass of a batch: per member the largest speed, the particles
with a non-finite component and those off the grid, for members smaller and
larger than the runs of slots that its workgroups take."""
from __future__ import annotations

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd import scenes
from mpm_amd.batch import Batch
from mpm_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1, 255, 256, 257, 5000, 1), (700_000, 3, 64, 130_000, 1, 1)])
def test_health_counts_every_member(sizes):
    solvers, want = [], []
    b = Batch(N.QUADRATIC_BSPLINE, N.PIC_FLIP)
    r = np.random.default_rng(len(sizes))
    for i, n in enumerate(sizes):
        sc = scenes.snow_cube(seed=i, n=n, res=32, transfer=N.PIC_FLIP)
        solvers.append(Solver(sc.desc, sc.particles))
        b.add(solvers[-1])
    for i, (n, s) in enumerate(zip(sizes, solvers)):
        st = s.read_particles()
        st.velocity[:] = r.normal(0, 1, (n, 3)).astype(np.float32)
        off = r.choice(n, n // 3, replace=False)  # two grids away
        st.position[off, i % 3] = 3.0
        bad = r.choice(n, min(n // 5, 7), replace=False)
        st.velocity[bad, 1] = np.inf if i % 2 else np.nan
        v = st.velocity
        sq = (v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1]) + v[:, 2] * v[:, 2]
        want.append((float(np.sqrt(np.float64(sq.max()))), len(bad), len(off)))
        s.write_particles(st)
    for got, (speed, bad, off) in zip(b.health(), want):
        assert (got["nonfinite"], got["escaped"]) == (bad, off)
        # the device may contract a product and a sum: two roundings of the square
        assert got["max_speed"] == speed or abs(got["max_speed"] - speed) <= 2.0**-23 * speed or (
            np.isnan(got["max_speed"]) and np.isnan(speed))
    b.close()
    for s in solvers:
        s.close()
