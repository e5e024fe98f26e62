"""P2G of the cubic stencil, term by term: a finite affine velocity whose
products overflow stays in its component, and the forces agree with the 64-bit
oracle where the elastic strain is large enough that 32 bits hold it."""
from __future__ import annotations

import numpy as np
import pytest

from mpm_amd import native as N
from mpm_amd.solver import Solver
from oracle import pyoracle
from tests.helpers import grid_errors, report
from tests.test_gpu_p2g_cubic import _desc, _state

pytestmark = pytest.mark.gpu


def _grids(d, st):
    gpu = Solver(d, st.copy(), run_initialize=False)
    ref = pyoracle.OracleSolver(d, st.copy(), 64, run_initialize=False)
    gpu.resetGrid()
    gpu.particlesToGrid()
    ref.substep("reset")
    ref.substep("p2g")
    return gpu.read_grid(), ref.read_grid()


def test_overflow_stays_in_its_component():
    # B_xy 1e35: C = 3 / h^2 B is finite, m C dx of a mass of 1e8 is not
    st, d = _state((40, 33, 5, 9), N.APIC), _desc(N.APIC)
    odd = 35
    st.B[odd] = 0.0
    st.mass[odd] = 1e8
    st.B[odd, 0, 1] = 1e35
    g, _ = _grids(d, st)
    st.B[odd, 0, 1] = 0.0
    _, r = _grids(d, st)
    assert np.isfinite(g["mass"]).all() and np.isfinite(g["force"]).all()
    p, q = g["velocity"].reshape(-1, 3), np.asarray(r["velocity"]).reshape(-1, 3)
    assert 0 < (~np.isfinite(p[:, 0])).sum() <= 64
    e = grid_errors(g, r, ("mass",))
    e["momentum yz"] = float(np.abs(p[:, 1:] - q[:, 1:]).max() / np.abs(q).max())
    report("cubic P2G, one overflow", e)
    assert all(v <= 1e-5 for v in e.values()), e


@pytest.mark.parametrize("transfer", [N.PIC_FLIP, N.APIC])
@pytest.mark.parametrize("counts", [(1,), (33, 31), (65, 64), (200, 3, 700, 1, 40, 5, 1)], ids=str)
def test_forces_of_a_large_strain(transfer, counts):
    # |Fe - R| ~ 0.3: its 32-bit rounding is 2^-24 / 0.3 of it, and a node's
    # force sums up to 1,000 of them; the bar is the parity bar, 1e-5 normwise
    st, d = _state(counts, transfer), _desc(transfer)
    r = np.random.default_rng(8)
    n = st.count
    st.Fe[:] = (np.diag([1.3, 0.8, 1.1]) + r.normal(0, 0.05, (n, 3, 3))).astype(np.float32)
    g, ref = _grids(d, st)
    e = grid_errors(g, ref, ("mass", "velocity", "force"))
    report(f"cubic P2G, large strain, {counts} {'APIC' if transfer else 'PIC-FLIP'}", e)
    assert np.abs(np.asarray(ref["force"])).max() > 0
    assert all(v <= 1e-5 for v in e.values()), e
