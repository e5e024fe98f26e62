"""What this solver is used for, as measurable cases.

Each case is one pass of a user's program over scenes that already live on the
device (or, for a restart, over a checkpoint in host memory): some steps, then
what that program takes out of them.  ``listed()`` names the cases, ``draw()``
gives more of the same ranges, ``prepare()`` builds the scenes, ``run()`` is the
pass, ``work()`` the bytes and operations it cannot do without, and ``exact()``
the same pass in 64 bits with plain torch.

The scenes are the workloads of the benchmark and the tests (snow cube, two
balls, jittered slab, unions of spheres and boxes) at their own and at odd
sizes; the snow material is the reference configuration's.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mpm_amd import native as N
from mpm_amd.batch import Batch
from mpm_amd.solver import ParticleInput, ParticleState, Solver, SolverDesc

RHO, E0, NU, XI, THETA_C, THETA_S = 400.0, 1.4e5, 0.2, 10.0, 2.5e-2, 7.5e-3
FRICTION, BLEND, GRAVITY = 0.9, 0.95, 9.8
EPS = 1.1920928955078125e-07  # FLT_EPSILON of the reference's conditions

PIC, APIC = N.PIC_FLIP, N.APIC
LIN, QUAD, CUB = N.LINEAR, N.QUADRATIC_BSPLINE, N.CUBIC_BSPLINE
WIDTH = {LIN: 2, QUAD: 3, CUB: 4}


def _case(name, use, shape, n, res, transfer, interp, steps, dt=1e-4, **more):
    """use: what the pass takes out ("state": the whole particle state on the
    host, "positions": (x, y, z, 1) in a device vertex buffer, "density": the
    raster's blocks on the host, "restart": a scene built from a checkpoint,
    stepped, read back and freed, "batch": many scenes stepped together)."""
    c = dict(name=name, use=use, shape=shape, n=n, rx=res[0], ry=res[1], rz=res[2], transfer=transfer, interp=interp,
             steps=steps, dt=dt, speed=0.0, young=1.0, model=N.FIXED_COROTATED, collide=False, graph=False, scenes=1,
             n_lo=0)
    c.update(more)
    return c


def listed():
    return [
        # The demo loop: one step per displayed frame of the small snow cube,
        # its vertex buffer filled on the device.  The smallest call; latency.
        _case("cube_frame", "positions", "cube", 16384, (64,) * 3, PIC, QUAD, 1),
        # The reference's CPU-runnable configuration, 50 steps and its state.
        _case("cube_run", "state", "cube", 16384, (64,) * 3, PIC, QUAD, 50),
        # The small cube as APIC, replayed as a captured step (programs that
        # capture their frame loop).
        _case("cube_graph", "state", "cube", 16384, (64,) * 3, APIC, QUAD, 50, graph=True, speed=1.0),
        # Linear weights, the other constitutive model, particles checked
        # against the walls: every option that a configuration can set.
        _case("linear_run", "state", "cube", 50021, (64,) * 3, PIC, LIN, 20, speed=0.5, model=N.NEO_HOOKEAN,
              collide=True),
        # The two colliding balls: cubic weights, 8 particles per cell.
        _case("balls_run", "state", "balls", 0, (128,) * 3, APIC, CUB, 50, dt=5e-5, speed=3.0),
        # A union of primitives with odd counts on an uneven odd-sized grid.
        _case("union_run", "state", "union", 290417, (101, 90, 111), APIC, QUAD, 50, speed=1.0),
        # Offline frames: a million particles, PIC-FLIP, the density raster
        # after every other step.
        _case("density_frame", "density", "slab", 1048576, (128,) * 3, PIC, QUAD, 2, dt=2.5e-5, speed=0.5),
        # A long run resumed from a checkpoint and saved again.
        _case("restart", "restart", "union", 120011, (128,) * 3, APIC, QUAD, 20, speed=1.0),
        # PIC-FLIP at production size.
        _case("slab_flip", "positions", "slab", 2097152, (160,) * 3, PIC, QUAD, 20, dt=2.5e-5, speed=0.5, young=4.0),
        # The headline workload: 8.4M particles, 256^3, APIC.
        _case("slab", "positions", "slab", 8388608, (256,) * 3, APIC, QUAD, 20, dt=2.5e-5, speed=0.5, young=4.0),
        # One server tick of PIC-FLIP requests of 5k to 500k particles.
        _case("served_tick", "batch", "union", 500000, (0,) * 3, PIC, QUAD, 16, speed=1.0, scenes=24, n_lo=5000),
        # The uneven batch: 256 scenes of 2k to 200k particles, APIC.
        _case("uneven_batch", "batch", "union", 200000, (0,) * 3, APIC, QUAD, 10, speed=1.0, scenes=256, n_lo=2000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    transfer = rng.choice([PIC, APIC])
    interp = rng.choice([QUAD, QUAD, CUB] if transfer == APIC else [LIN, QUAD, QUAD, CUB])
    use = rng.choice(["positions", "state", "state", "density", "restart", "batch"])
    steps = rng.randint(1, 40)
    if use == "batch":
        return _nameless(_case("", "batch", "union", _log(rng, 20000, 300000), (0,) * 3, transfer, interp, min(steps, 16),
                               speed=1.0, scenes=_log(rng, 3, 64), n_lo=_log(rng, 1000, 8000)))
    n = _log(rng, 2000, 400000 if use in ("state", "restart") else 3000000)
    # about 2 to 8 particles per cell, in up to a third of the domain
    cells = n / math.exp(rng.uniform(math.log(2.0), math.log(8.0)))
    r = min(256, max(24, int((cells / 0.1) ** (1 / 3))))
    res = tuple(r + rng.randint(-3, 3) for _ in range(3))
    shape = rng.choice(["cube", "slab", "union"])
    return _nameless(_case("", use, shape, n, res, transfer, interp, 2 if use == "density" else steps,
                           dt=min(1e-4, 0.006 / r), speed=rng.choice([0.25, 0.5, 1.0]), young=rng.choice([1.0, 4.0]),
                           model=rng.choice([N.FIXED_COROTATED] * 3 + [N.NEO_HOOKEAN]), collide=rng.random() < 0.25,
                           graph=use == "state" and rng.random() < 0.25))


def _nameless(c):
    del c["name"]
    return c


# ------------------------------------------------------------------- inputs
def _union(r, n, center, extent):
    """n points uniform in a union of 1-4 spheres and boxes, and its volume:
    points of the single shapes, each kept with 1 / (shapes that hold it)."""
    shapes = [(int(r.integers(0, 2)), center + r.uniform(-0.2, 0.2, 3) * extent, extent * r.uniform(0.15, 0.3))
              for _ in range(int(r.integers(1, 5)))]
    volume = np.array([(4 / 3 * math.pi if ball else 8.0) * s ** 3 for ball, _, s in shapes])
    got, tried, kept = [], 0, 0
    while kept < n:
        m = int(1.2 * (n - kept)) + 64
        p = []
        for k, (ball, c, s) in zip(r.multinomial(m, volume / volume.sum()), shapes):
            d = r.uniform(-1, 1, (2 * k + 64 if ball else k, 3))
            p.append(c + s * (d[(d * d).sum(1) <= 1.0][:k] if ball else d))
        p = r.permutation(np.concatenate(p))
        held = sum((((p - c) ** 2).sum(1) <= s * s if ball else (np.abs(p - c) <= s).all(1)).astype(np.int64)
                   for ball, c, s in shapes)
        got.append(p[r.random(len(p)) * held < 1.0])
        tried += len(p)
        kept += len(got[-1])
    return np.concatenate(got)[:n], float(volume.sum()) * kept / tried


def _thrown(r, d, speed):
    """Velocities of a body thrown with a spin; d: places about its centre."""
    return speed * (r.uniform(-1, 1, 3) + np.cross(r.uniform(-4, 4, 3), d))


def _scene(case, r, n, res):
    """One scene's grid and particles (positions, velocity, mass, young)."""
    h = 1.0 / res[0]
    size = np.array(res) * h
    if case["shape"] == "cube":
        # the benchmark cube's density: 7.8 particles per cell at 16384 in 64^3
        side = min(0.8, (n / 7.8) ** (1 / 3) * h)
        pos = 0.5 * size + (r.random((n, 3)) - 0.5) * side * size
        volume = side ** 3 * float(np.prod(size))
        vel = _thrown(r, pos - pos.mean(0), case["speed"])
    elif case["shape"] == "balls":
        rad, ppc = 0.1, 8
        n = int(4 / 3 * math.pi * rad ** 3 / h ** 3 * ppc)
        d = r.normal(size=(2 * n, 3))
        d *= (rad * r.random(2 * n) ** (1 / 3) / np.sqrt((d * d).sum(1)))[:, None]
        left = np.arange(2 * n) < n
        pos = d + np.where(left[:, None], (0.3, 0.5, 0.5), (0.7, 0.5, 0.5))
        vel = np.where(left, case["speed"], -case["speed"])[:, None] * np.array([1.0, 0.0, 0.0])
        vel = vel + np.cross(np.where(left[:, None], *r.uniform(-8, 8, (2, 3))), d)
        n, volume = 2 * n, 2 * n * h ** 3 / ppc
    elif case["shape"] == "slab":
        # a jittered lattice, twice as wide as high, normal velocities
        ny = max(1, int(round((n / 4) ** (1 / 3))))
        count = np.array([2 * ny, ny, -(-n // (2 * ny * ny))])
        lo, hi = 0.1 * size, np.array([0.9, 0.5, 0.9]) * size
        at = np.indices(count[::-1], np.float32).reshape(3, -1)[::-1, :n].T
        pos = lo + (at + (0.25 + 0.5 * r.random((n, 3), np.float32))) * ((hi - lo) / count)
        volume = float(np.prod((hi - lo) / count)) * n
        vel = r.standard_normal((n, 3), np.float32) * case["speed"]
    else:
        pos, volume = _union(r, n, np.array([0.5, 0.45, 0.5]) * size, 0.4)
        vel = _thrown(r, pos - pos.mean(0), case["speed"])
    f = np.float32
    return dict(res=res, h=f(h), n=n, pos=pos.astype(f), vel=np.broadcast_to(vel, (n, 3)).astype(f),
                mass=f(RHO * volume / n), young=(E0 * r.uniform(1.0, case["young"], n)).astype(f))


def _scenes(case, seed):
    r = np.random.default_rng(seed)
    if case["use"] != "batch":
        return [_scene(case, r, case["n"], (case["rx"], case["ry"], case["rz"]))]
    out = []
    # sizes log-uniform in [n_lo, n], in a shuffled order
    u = (np.random.default_rng(3).permutation(case["scenes"]) + 0.5) / case["scenes"]
    for n in (case["n_lo"] * (case["n"] / case["n_lo"]) ** u).round().astype(int):
        res = 32 if n < 15000 else 64 if n < 60000 else 128 if n < 250000 else 256
        out.append(_scene(case, r, int(n), (res,) * 3))
    return out


def _desc(case, sc):
    return SolverDesc((0.0, 0.0, 0.0), sc["res"], float(sc["h"]), FRICTION, BLEND, case["interp"], case["transfer"],
                      case["dt"], GRAVITY, case["collide"])


def _particles(case, sc):
    return ParticleInput(sc["pos"], sc["vel"], sc["mass"], XI, sc["young"], NU, THETA_C, THETA_S, case["model"])


def _checkpoint(case, sc, seed):
    """A state in the middle of a run: deformed within and beyond the
    thresholds, some of it plastic."""
    r = np.random.default_rng([seed, 7])
    n, f = sc["n"], np.float32
    e = sc["young"].astype(np.float64)
    eye = np.eye(3)
    return ParticleState(
        volume0=np.full(n, float(sc["mass"]) / RHO, f), mass=np.full(n, sc["mass"], f), position=sc["pos"],
        velocity=sc["vel"] + r.normal(0, 0.05, (n, 3)).astype(f),
        Fe=(eye + r.normal(0, 0.003, (n, 3, 3))).astype(f), Fp=(eye + r.normal(0, 0.01, (n, 3, 3))).astype(f),
        mu0=(e / (2 * (1 + NU))).astype(f), lambda0=(e * NU / ((1 + NU) * (1 - 2 * NU))).astype(f),
        hardening=np.full(n, XI, f), critical_compression=np.full(n, THETA_C, f),
        critical_stretch=np.full(n, THETA_S, f), model=np.full(n, case["model"], np.int32),
        B=(r.normal(0, 0.05, (n, 3, 3)) * float(sc["h"])).astype(f) if case["transfer"] == APIC else None)


def prepare(case, seed):
    scenes = _scenes(case, seed)
    state = dict(case=case)
    if case["use"] == "restart":
        return dict(state, desc=_desc(case, scenes[0]), checkpoint=_checkpoint(case, scenes[0], seed))
    state["solvers"] = [Solver(_desc(case, sc), _particles(case, sc)) for sc in scenes]
    if case["use"] == "batch":
        state["batch"] = Batch(case["interp"], case["transfer"])
        for s in state["solvers"]:
            state["batch"].add(s)
    if case["use"] in ("positions", "batch"):
        counts = [s.count for s in state["solvers"]]
        buf = torch.empty(sum(counts), 4, device="cuda")
        state["vertices"] = buf
        state["pointers"] = [buf.data_ptr() + 16 * int(k) for k in np.cumsum([0] + counts[:-1])]
        torch.cuda.synchronize()
    return state


def _state_of(s):
    st = s.read_particles()
    out = {k: getattr(st, k) for k in ("volume0", "mass", "position", "velocity", "Fe", "Fp", "mu0", "lambda0")}
    if st.B is not None:
        out["B"] = st.B
    return out


def run(state):
    case = state["case"]
    if case["use"] == "restart":
        s = Solver(state["desc"], state["checkpoint"], run_initialize=False)
        s.step(case["steps"])
        out = _state_of(s)
        s.close()
        return out
    if case["use"] == "batch":
        b = state["batch"]
        b.step(case["steps"])
        for s, p in zip(state["solvers"], state["pointers"]):
            s.pack_positions4(p)
        # the server's check after a tick, which waits for it; the first
        # member is read back whole, as one whose request is done
        health = b.health()
        done = _state_of(state["solvers"][0])
        return {"vertices": state["vertices"], "done": done,
                **{k: np.array([h[k] for h in health]) for k in ("max_speed", "cfl", "nonfinite", "escaped")}}
    s = state["solvers"][0]
    (s.step_graph if case["graph"] else s.step)(case["steps"])
    if case["use"] == "state":
        return _state_of(s)
    if case["use"] == "density":
        return s.density()
    # the pack is asynchronous on the solver's own stream: the buffer may be
    # drawn from after this wait
    s.pack_positions4(state["pointers"][0])
    s.synchronize()
    return state["vertices"]


def work(case):
    """Per particle-step the state streamed once (APIC 280 B, PIC-FLIP 208 B;
    x, v, B, Fe, Fp read and written, m, V0, mu0, lambda0 read), per active
    node mass and momentum written once and read once, and the outputs."""
    if case["use"] == "batch":
        n = case["scenes"] * (case["n"] - case["n_lo"]) / math.log(case["n"] / case["n_lo"])
    elif case["shape"] == "balls":
        n = 2 * (4 / 3 * math.pi * 0.1 ** 3 * 8) * case["rx"] ** 3
    else:
        n = case["n"]
    w3 = WIDTH[case["interp"]] ** 3
    per = 280 if case["transfer"] == APIC else 208
    nodes = n / 2 if case["shape"] == "slab" else n / 5
    out = {"state": 200, "restart": 360, "density": 4, "positions": 16, "batch": 16}[case["use"]]
    # gather (v, grad v, B) and scatter (mass, momentum, force) per node;
    # weights, F update and stress per particle
    flops = case["steps"] * n * (w3 * (2 * 9 + 2 * 8) + 600)
    return {"bytes": case["steps"] * (n * per + nodes * 32) + n * out, "flops": flops}


# ------------------------------------------------------------ 64-bit result
def _svd3(a):
    """Singular value decomposition of n 3x3 matrices (3, 3, n) by cyclic
    Jacobi on A^T A: U (3, 3, n), s (3, n) with the sign of det A on the
    smallest, V (3, 3, n) with A = U diag(s) V^T."""
    s = [[(a[:, i] * a[:, j]).sum(0) for j in range(3)] for i in range(3)]
    v = [[torch.full_like(s[0][0], float(i == j)) for j in range(3)] for i in range(3)]
    for _ in range(6):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            r = 3 - p - q
            d = s[q][q] - s[p][p]
            den = d.abs() + torch.sqrt(d * d + 4 * s[p][q] ** 2)
            t = torch.where(den > 0, torch.where(d >= 0, 2.0, -2.0) * s[p][q] / den.clamp_min(1e-300), 0.0)
            c = 1 / torch.sqrt(1 + t * t)
            w = t * c
            s[p][p], s[q][q] = s[p][p] - t * s[p][q], s[q][q] + t * s[p][q]
            s[p][q] = s[q][p] = torch.zeros_like(t)
            s[r][p], s[r][q] = c * s[r][p] - w * s[r][q], w * s[r][p] + c * s[r][q]
            s[p][r], s[q][r] = s[r][p], s[r][q]
            for k in range(3):
                v[k][p], v[k][q] = c * v[k][p] - w * v[k][q], w * v[k][p] + c * v[k][q]
    V = torch.stack([torch.stack(row) for row in v])
    AV = _mm(a, V)
    sv = torch.sqrt((AV * AV).sum(0))
    U = AV / sv
    # a reflection goes to the smallest value
    flip = (torch.arange(3, device=sv.device)[:, None] == sv.argmin(0)) & (_det(a) < 0)
    sign = torch.where(flip, -1.0, 1.0)
    return U * sign, sv * sign, V


def _mm(a, b):
    return torch.stack([torch.stack([a[i, 0] * b[0, j] + a[i, 1] * b[1, j] + a[i, 2] * b[2, j] for j in range(3)])
                        for i in range(3)])


def _det(a):
    return (a[0, 0] * (a[1, 1] * a[2, 2] - a[1, 2] * a[2, 1]) - a[0, 1] * (a[1, 0] * a[2, 2] - a[1, 2] * a[2, 0]) +
            a[0, 2] * (a[1, 0] * a[2, 1] - a[1, 1] * a[2, 0]))


def _weights(interp, d):
    """B-spline weight and derivative at offset d (in cells)."""
    x, sg = d.abs(), torch.sign(d)
    if interp == LIN:
        return torch.where(x < 1, 1 - x, 0.0), torch.where((x < 1) & (x > EPS), -sg, 0.0)
    if interp == QUAD:
        return (torch.where(x < 0.5, 0.75 - x * x, torch.where(x < 1.5, 0.5 * (1.5 - x) ** 2, 0.0)),
                torch.where(x < 0.5, -2 * d, torch.where(x < 1.5, d - 1.5 * sg, 0.0)))
    return (torch.where(x < 1, 0.5 * x ** 3 - x * x + 2 / 3, torch.where(x < 2, (2 - x) ** 3 / 6, 0.0)),
            torch.where(x < 1, 1.5 * d * x - 2 * d, torch.where(x < 2, 2 * d - 2 * sg - 0.5 * d * x, 0.0)))


class _Exact:
    """The step in 64 bits over the particles of all scenes at once; vectors
    are (3, n) and matrices (3, 3, n)."""

    def __init__(self, case, scenes, seed):
        self.case, self.scenes = case, scenes
        f64 = dict(dtype=torch.float64, device="cuda")
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), **f64)  # noqa: E731
        per = lambda key: t(np.concatenate([np.full(s["n"], float(key(s))) for s in scenes]))  # noqa: E731
        self.n = sum(s["n"] for s in scenes)
        self.dt, self.g = float(np.float32(case["dt"])), float(np.float32(GRAVITY))
        self.mu_b, self.blend = float(np.float32(FRICTION)), float(np.float32(BLEND))
        self.hi, self.lo = 1 + float(np.float32(THETA_S)), 1 - float(np.float32(THETA_C))
        self.apic, self.W = case["transfer"] == APIC, WIDTH[case["interp"]]
        self.x = t(np.concatenate([s["pos"] for s in scenes]).T)
        self.v = t(np.concatenate([s["vel"] for s in scenes]).T)
        self.m = per(lambda s: s["mass"])
        self.h = per(lambda s: s["h"])
        sizes = [int(np.prod(s["res"])) for s in scenes]
        self.first = np.cumsum([0] + sizes)
        index = np.repeat(np.arange(len(scenes)), [s["n"] for s in scenes])
        to = lambda a: torch.as_tensor(np.asarray(a)[index], device="cuda")  # noqa: E731
        self.off = to(self.first[:-1].astype(np.int64))
        self.res = [to(np.array([s["res"][k] for s in scenes], np.int64)) for k in range(3)]
        if case["use"] == "restart":
            c = _checkpoint(case, scenes[0], seed)
            self.V0, self.mu0, self.la0, self.v = t(c.volume0), t(c.mu0), t(c.lambda0), t(c.velocity.T)
            self.Fe, self.Fp = (t(a.transpose(1, 2, 0)) for a in (c.Fe, c.Fp))
            self.B = t(c.B.transpose(1, 2, 0)) if self.apic else None
        else:
            e, nu = t(np.concatenate([s["young"] for s in scenes])), float(np.float32(NU))
            self.mu0, self.la0 = e / (2 * (1 + nu)), e * nu / ((1 + nu) * (1 - 2 * nu))
            self.Fe = torch.eye(3, **f64)[:, :, None].repeat(1, 1, self.n)
            self.Fp = self.Fe.clone()
            self.B = torch.zeros_like(self.Fe) if self.apic else None
            self.V0 = self.m * self.h ** 3 / self._gather_mass(self._scatter_mass())
        # target corner and node position of each grid node of every scene
        self.node_h = torch.repeat_interleave(t([float(s["h"]) for s in scenes]), torch.tensor(sizes, device="cuda"))

    def _axes(self):
        """Base node and per-axis weights of the current positions."""
        u = self.x / self.h
        base = torch.floor(u - 0.5 * (self.W - 2))
        N_, D_ = zip(*[_weights(self.case["interp"], u - (base + j)) for j in range(self.W)])
        return base.long(), N_, D_

    def _nodes(self, base):
        """(a, b, c), linear index and in-grid mask of every stencil node."""
        W = self.W
        for a in range(W):
            for b in range(W):
                for c in range(W):
                    i, j, k = base[0] + a, base[1] + b, base[2] + c
                    ok = ((i >= 0) & (i < self.res[0]) & (j >= 0) & (j < self.res[1]) & (k >= 0) & (k < self.res[2]))
                    q = self.off + i + self.res[0] * (j + self.res[1] * k)
                    yield a, b, c, torch.where(ok, q, 0), ok.to(torch.float64)

    def _scatter_mass(self):
        base, N_, _ = self._axes()
        mass = torch.zeros(int(self.first[-1]), dtype=torch.float64, device="cuda")
        for a, b, c, q, ok in self._nodes(base):
            mass.index_add_(0, q, ok * self.m * N_[a][0] * N_[b][1] * N_[c][2])
        return mass

    def _gather_mass(self, mass):
        base, N_, _ = self._axes()
        out = torch.zeros_like(self.m)
        for a, b, c, q, ok in self._nodes(base):
            out += ok * mass[q] * N_[a][0] * N_[b][1] * N_[c][2]
        return out

    def _walls(self, p, v, corner):
        """The reference's boundary collision of velocities v at p."""
        n = torch.zeros_like(v)
        for k in range(3):
            n[k] = torch.where(p[k] >= corner[k] - EPS, -1.0, torch.where(p[k] <= EPS, 1.0, 0.0))
        vn = (v * n).sum(0)
        vt = v - vn * n
        nt = torch.sqrt((vt * vt).sum(0))
        slide = vt + self.mu_b * vn * vt / nt.clamp_min(1e-300)
        new = torch.where(nt <= -self.mu_b * vn + EPS, 0.0, slide)
        return torch.where((n != 0).any(0) & (vn < EPS), new, v)

    def _stress(self):
        """-V0 P Fe^T."""
        U, s, _ = _svd3(self.Fe)
        f = torch.exp(float(np.float32(XI)) * (1 - _det(self.Fp)))
        mu, la = self.mu0 * f, self.la0 * f
        J = s.prod(0)
        if self.case["model"] == N.NEO_HOOKEAN:
            d, c = mu * (s * s - 1), la * torch.log(J)
        else:
            d, c = 2 * mu * (s - 1) * s, la * (J - 1) * J
        return -self.V0 * _mm(U * (d + c), U.transpose(0, 1))

    def step(self):
        tau = self._stress()
        base, N_, D_ = self._axes()
        x, h, W = self.x, self.h, self.W
        grid = torch.zeros(int(self.first[-1]), 7, dtype=torch.float64, device="cuda")
        C = self.B * ((4 if self.case["interp"] == QUAD else 3) / h ** 2) if self.apic else None
        for a, b, c, q, ok in self._nodes(base):
            nx, ny, nz = N_[a][0], N_[b][1], N_[c][2]
            g = torch.stack([D_[a][0] * ny * nz, nx * D_[b][1] * nz, nx * ny * D_[c][2]]) / h
            mw = ok * self.m * nx * ny * nz
            v = self.v
            if self.apic:
                dx = torch.stack([(base[k] + e) * h - x[k] for k, e in enumerate((a, b, c))])
                v = v + (C * dx).sum(1)
            grid.index_add_(0, q, torch.cat([mw[None], mw * v, ok * (tau * g).sum(1)]).T.contiguous())
        m = grid[:, 0]
        heavy = m > EPS
        inv = torch.where(heavy, 1 / m.clamp_min(1e-300), 0.0)
        vel = torch.where(heavy, grid[:, 1:4].T * inv, grid[:, 1:4].T)
        f = grid[:, 4:7].T
        star = torch.where(heavy, vel + self.dt * f * inv, 0.0)
        star[1] -= torch.where(heavy, self.dt * self.g, 0.0)
        for s, lo, hi in zip(self.scenes, self.first[:-1], self.first[1:]):
            r = s["res"]
            i = torch.arange(int(hi - lo), device="cuda")
            node = torch.stack([i % r[0], i // r[0] % r[1], i // (r[0] * r[1])]) * float(s["h"])
            st = star[:, int(lo):int(hi)]
            star[:, int(lo):int(hi)] = self._walls(node + self.dt * st, st, [float(s["h"]) * k for k in r])
        del grid, f, inv, heavy
        table = torch.cat([star, star - vel]).T.contiguous()
        del star, vel
        pic, flip = torch.zeros_like(x), self.v.clone()
        grad, B = torch.zeros_like(self.Fe), torch.zeros_like(self.Fe)
        for a, b, c, q, ok in self._nodes(base):
            nx, ny, nz = N_[a][0], N_[b][1], N_[c][2]
            g = torch.stack([D_[a][0] * ny * nz, nx * D_[b][1] * nz, nx * ny * D_[c][2]]) / h
            w = nx * ny * nz
            val = table[q].T * ok
            pic += w * val[:3]
            flip += w * val[3:]
            grad += val[:3, None] * g
            if self.apic:
                dx = torch.stack([(base[k] + e) * h - x[k] for k, e in enumerate((a, b, c))])
                B += w * val[:3, None] * dx
        self.v = pic if self.apic else self.blend * flip + (1 - self.blend) * pic
        if self.apic:
            self.B = B
        if self.case["collide"]:
            self.v = self._walls(x + self.dt * self.v, self.v, [h * r for r in self.res])
        self.x = x + self.dt * self.v
        eye = torch.eye(3, dtype=torch.float64, device="cuda")[:, :, None]
        Fn = _mm(eye + self.dt * grad, self.Fe)
        U, s, V = _svd3(Fn)
        sc = s.clamp(self.lo, self.hi)
        self.Fp = _mm(_mm(V * (s / sc), V.transpose(0, 1)), self.Fp)
        self.Fe = _mm(U * sc, V.transpose(0, 1))

    def positions(self):
        return torch.cat([self.x, torch.ones_like(self.x[:1])]).T.contiguous()

    def state(self, n):
        mat = lambda a: a[:, :, :n].permute(2, 0, 1).contiguous()  # noqa: E731
        out = dict(volume0=self.V0[:n], mass=self.m[:n], position=self.x[:, :n].T.contiguous(),
                   velocity=self.v[:, :n].T.contiguous(), Fe=mat(self.Fe), Fp=mat(self.Fp), mu0=self.mu0[:n],
                   lambda0=self.la0[:n])
        if self.apic:
            out["B"] = mat(self.B)
        return out

    def density(self):
        return self._scatter_mass() / float(self.scenes[0]["h"]) ** 3


def exact(case, seed):
    scenes = _scenes(case, seed)
    if sum(s["n"] for s in scenes) * case["steps"] * WIDTH[case["interp"]] ** 3 > 6e9:
        return None  # too long
    e = _Exact(case, scenes, seed)
    for _ in range(case["steps"]):
        e.step()
    if case["use"] in ("state", "restart"):
        return e.state(e.n)
    if case["use"] == "density":
        return e.density()
    if case["use"] == "positions":
        return e.positions()
    speed = [float(torch.sqrt((v * v).sum(0).amax())) for v in e.v.split([s["n"] for s in scenes], 1)]
    return {"vertices": e.positions(), "done": e.state(scenes[0]["n"]), "max_speed": np.array(speed),
            "cfl": np.array([v * e.dt / float(s["h"]) for v, s in zip(speed, scenes)]), "nonfinite": None,
            "escaped": None}
