"""P2G of the cubic stencil (cell sums on the matrix cores) at the sizes where
it can go wrong: cells of one particle, of a record batch (32), a wave (64),
an item and their neighbours, cells at tile corners, and particles whose
affine velocity is not finite."""
from __future__ import annotations

from dataclasses import fields

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd.solver import ParticleState, Solver, SolverDesc
from oracle import pyoracle
from tests.helpers import grid_errors, particle_errors, rel_err, report

pytestmark = pytest.mark.gpu

RES = 20


def _state(counts, transfer, seed=3):
    """counts[k] particles in the k-th of some cells (block corners first),
    deformed, with velocities of one sign (no cancellation in the sums)."""
    r = np.random.default_rng(seed)
    cells = [(3, 3, 3), (4, 4, 4), (7, 7, 7), (8, 7, 4), (5, 6, 7), (6, 6, 7), (11, 4, 8)]
    pos = np.concatenate([(np.array(c) + 1.0 + r.uniform(0.05, 0.95, (k, 3))) / RES for c, k in zip(cells, counts)])
    n = len(pos)
    f = np.float32
    return ParticleState(
        volume0=np.full(n, 1e-6, f), mass=r.uniform(0.5, 1.5, n).astype(f) * f(1e-3), position=pos.astype(f),
        velocity=r.uniform(0.5, 1.5, (n, 3)).astype(f), Fe=(np.eye(3) + r.normal(0, 0.004, (n, 3, 3))).astype(f),
        Fp=(np.eye(3) + r.normal(0, 0.01, (n, 3, 3))).astype(f), mu0=np.full(n, 6e4, f), lambda0=np.full(n, 4e4, f),
        hardening=np.full(n, 10, f), critical_compression=np.full(n, 0.025, f), critical_stretch=np.full(n, 0.0075, f),
        model=np.zeros(n, np.int32),
        B=(r.normal(0, 0.1, (n, 3, 3)) / RES).astype(f) if transfer == N.APIC else None)


def _part(st, which):
    return ParticleState(**{f.name: None if getattr(st, f.name) is None else getattr(st, f.name)[which].copy()
                            for f in fields(ParticleState)})


def _desc(transfer):
    return SolverDesc(resolution=(RES,) * 3, stride=1 / RES, transfer=transfer, interp=N.CUBIC_BSPLINE, dt=1e-4)


@pytest.mark.parametrize("transfer", [N.PIC_FLIP, N.APIC])
@pytest.mark.parametrize("counts", [(1,), (31, 2), (32,), (33, 31), (63, 1, 2), (65, 64), (200, 3, 700, 1, 40, 5, 1)],
                         ids=str)
def test_cell_sums(counts, transfer):
    # the grid of the sub-step and the particles after a step (APIC: the
    # folded sums), at the parity bar (1e-5 normwise)
    st, d = _state(counts, transfer), _desc(transfer)
    gpu = Solver(d, st.copy(), run_initialize=False)
    ref = pyoracle.OracleSolver(d, st.copy(), 64, run_initialize=False)
    gpu.resetGrid()
    gpu.particlesToGrid()
    ref.substep("reset")
    ref.substep("p2g")
    g = gpu.read_grid()
    e = grid_errors(g, ref.read_grid(), ("mass", "velocity"))
    # the force, whose value is only as good as FP32 holds Fe - R (|Fe - R|
    # ~ 1e-2 here), against the sum of the two halves' own forces
    halves = []
    for k in range(2):
        part = _part(st, slice(k, None, 2))
        s = Solver(d, part, run_initialize=False)
        s.resetGrid()
        s.particlesToGrid()
        halves.append(s.read_grid()["force"].astype(np.float64))
    e["force"] = rel_err(g["force"], halves[0] + halves[1])
    gpu.step(1)
    ref2 = pyoracle.OracleSolver(d, st.copy(), 64, run_initialize=False)
    ref2.step(1)
    e.update(particle_errors(gpu.read_particles(), ref2.read_particles()))
    report(f"cubic P2G {counts} {'APIC' if transfer else 'PIC-FLIP'}", e)
    assert all(v <= 1e-5 for v in e.values()), e


def test_non_finite_particle_stays_in_its_components():
    # an infinite B_xy: only the x momentum of its own 64 nodes may be lost
    st, d = _state((40, 33, 5, 9), N.APIC), _desc(N.APIC)
    odd = 35
    st.B[odd] = 0.0
    clean = pyoracle.OracleSolver(d, st.copy(), 64, run_initialize=False)
    same = Solver(d, st.copy(), run_initialize=False)
    st.B[odd, 0, 1] = np.inf
    gpu = Solver(d, st, run_initialize=False)
    gpu.resetGrid()
    gpu.particlesToGrid()
    same.resetGrid()
    same.particlesToGrid()
    clean.substep("reset")
    clean.substep("p2g")
    g, r = gpu.read_grid(), clean.read_grid()
    for k in ("mass", "force"):
        assert np.isfinite(g[k]).all()
    e = grid_errors(g, r, ("mass",))
    e["force"] = rel_err(g["force"], same.read_grid()["force"])
    p, q = g["velocity"].reshape(-1, 3), np.asarray(r["velocity"]).reshape(-1, 3)
    e["momentum yz"] = float(np.abs(p[:, 1:] - q[:, 1:]).max() / np.abs(q).max())
    lost = ~np.isfinite(p[:, 0])
    assert 0 < lost.sum() <= 64
    e["momentum x"] = float(np.abs(p[~lost, 0] - q[~lost, 0]).max() / np.abs(q).max())
    report("cubic P2G, one infinite B", e)
    assert all(v <= 1e-5 for v in e.values()), e
