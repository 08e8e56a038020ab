"""The framework's work as its users have it do: runs through the public entry points.

A case names a family and its sizes:

* ``wave``      1-D periodic acoustic wave, forward + discrete adjoint with the control
                gradient (a member of the mixed batches; the smallest grids there are).
* ``monopole``  2-D acoustic monopole on an odd square grid with sponges, far field and a
                control; ``forward`` alone (the line search and the finite-difference sweep:
                the instances are the amplitudes) or ``adjoint`` (a gradient evaluation).
* ``loop``      the same monopole driven stage by stage by the caller's own time loop.
* ``shooting``  2-D mixing layer, multiple shooting: msforward + msadjoint, the segments
                being the instances of one region.
* ``ensemble``  small monopoles of different sizes, forward + adjoint, merged launches.
* ``flow``      3-D viscous periodic Kolmogorov flow; ``forward`` alone or ``adjoint`` from
                the terminal kinetic energy (the gradient with respect to the initial
                condition).  Grids of any size, not multiples of a tile only.

``exact`` is a plain torch model of the same discrete problem (dense SBP matrices,
automatic differentiation of the spatial operator), independent of the package.
"""
from __future__ import annotations

import dataclasses
import math
from fractions import Fraction

import numpy as np
import torch

from magudi_amd import cases as mc


# ---------------------------------------------------------------------------- the cases
def listed():
    return [
        # one 1-D member of a mixed batch: 2048 points, launch latency and nothing else
        {"name": "wave_2048_adjoint", "family": "wave", "n": 2048, "steps": 64, "save": 16},
        # a host program's own time loop over the stage entry points on a small odd grid,
        # with the functional after every stage as the Solver loop takes it
        {"name": "loop_101_forward", "family": "loop", "n": 101, "steps": 16},
        # one forward run of the basic configuration (201^2, half its 480 steps)
        {"name": "monopole_201_forward", "family": "monopole", "n": 201, "steps": 240,
         "save": 32, "instances": 1, "adjoint": False},
        # one gradient evaluation of the ordinary grid: forward, adjoint, control gradient
        {"name": "monopole_401_adjoint", "family": "monopole", "n": 401, "steps": 320,
         "save": 32, "instances": 1, "adjoint": True},
        # the finite-difference sweep: 20 control amplitudes as the instances of one region
        {"name": "sweep20_401_forward", "family": "monopole", "n": 401, "steps": 96,
         "save": 32, "instances": 20, "adjoint": False},
        # a batch of gradients on an odd grid
        {"name": "batch8_273_adjoint", "family": "monopole", "n": 273, "steps": 96,
         "save": 16, "instances": 8, "adjoint": True},
        # multiple shooting of the mixing layer, 4 segments of 32 steps
        {"name": "shooting4_513x257", "family": "shooting", "nx": 513, "ny": 257, "segments": 4,
         "steps": 32, "save": 8},
        # an ensemble of small grids of different sizes, one launch per stage for all
        {"name": "ensemble16_merged", "family": "ensemble", "members": 16, "lo": 41, "hi": 201,
         "steps": 32, "save": 8},
        # the 3-D flow on a small grid: a gradient with respect to the initial condition
        {"name": "flow_64_adjoint", "family": "flow", "n": 64, "steps": 16, "save": 4,
         "adjoint": True, "held": -1},
        # the same on a size that is no multiple of a tile
        {"name": "flow_100_adjoint", "family": "flow", "n": 100, "steps": 12, "save": 4,
         "adjoint": True, "held": -1},
        # a forward run of a mid-size 3-D grid
        {"name": "flow_160_forward", "family": "flow", "n": 160, "steps": 32, "save": 8,
         "adjoint": False, "held": -1},
        # the large flow, forward + adjoint; a third of the steps' stage states held and the
        # others recomputed, as in a 200-step run at this size
        {"name": "flow_256_adjoint", "family": "flow", "n": 256, "steps": 24, "save": 8,
         "adjoint": True, "held": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["wave", "loop", "monopole", "monopole", "monopole", "shooting",
                         "ensemble", "flow", "flow", "flow"])
    if family == "wave":
        steps = rng.randint(24, 64)
        return {"family": family, "n": _log_int(rng, 192, 4096), "steps": steps,
                "save": rng.randint(5, 16)}
    if family == "loop":
        return {"family": family, "n": 2 * rng.randint(20, 100) + 1, "steps": rng.randint(6, 20)}
    if family == "monopole":
        n = 2 * rng.randint(25, 256) + 1
        inst = rng.choice([1, 1, 2, 3, 5, 8, 13, 20])
        steps = _log_int(rng, 24, 240)
        steps = max(16, min(steps, int(1.2e8 / (n * n * inst))))
        return {"family": family, "n": n, "steps": steps, "save": rng.randint(7, 32),
                "instances": inst, "adjoint": rng.random() < 0.5}
    if family == "shooting":
        return {"family": family, "nx": rng.randint(96, 513), "ny": 2 * rng.randint(30, 128) + 1,
                "segments": rng.randint(2, 6), "steps": rng.randint(12, 32),
                "save": rng.randint(4, 9)}
    if family == "ensemble":
        return {"family": family, "members": rng.randint(4, 16), "lo": 41,
                "hi": 2 * rng.randint(40, 110) + 1, "steps": rng.randint(12, 36),
                "save": rng.randint(5, 9)}
    n = _log_int(rng, 32, 232)
    steps = max(4, min(24, int(1.6e8 / n ** 3)))
    adjoint = rng.random() < 0.6
    return {"family": "flow", "n": n, "steps": steps, "save": max(2, steps // 4),
            "adjoint": adjoint, "held": rng.choice([-1, -1, 1]) if adjoint else -1}


# ---------------------------------------------------------------- inputs, from the seed
def _pulses(case, rng, count, amplitude, width):
    """Quiescent (or target) state plus acoustic pulses p' = rho' at random places."""
    x = case.coords
    dp = np.zeros(case.npoints)
    for _ in range(count):
        r2 = np.zeros(case.npoints)
        for d in range(case.nd):
            lo, hi = x[d].min(), x[d].max()
            c = rng.uniform(lo + 0.25 * (hi - lo), hi - 0.25 * (hi - lo))
            r2 += ((x[d] - c) / (width * (hi - lo))) ** 2
        dp += amplitude * rng.uniform(0.5, 1.5) * np.exp(-r2)
    q = case.initial_state()
    q[0] += dp
    for d in range(case.nd):
        q[1 + d] += q[1 + d] / (q[0] - dp) * dp      # the velocity stays
    q[case.nd + 1] += dp / (case.gamma - 1.0)
    return q


def _control(rng, case, instances, stages):
    """Actuator forcing: a few random tones over the stages, random over the points."""
    pts = len(case.patch_points(case.patches_of(mc.ACTUATOR)[0]))
    s = np.arange(stages)[:, None] / stages
    out = np.empty((instances, stages, pts))
    shape = rng.standard_normal((3, pts))
    tones = [np.sin(2 * np.pi * ((k + 1) * s + rng.uniform())) for k in range(3)]
    base = sum(t * shape[k] for k, t in enumerate(tones))
    for i in range(instances):
        out[i] = 1e-2 * 10.0 ** (-0.25 * i) * base
    return out


def _monopole(n, steps, save, rng):
    """The cost annulus reaches in over the control, so that short runs have a gradient too."""
    c = mc.acoustic_monopole(n=n, nsteps=steps, save_interval=save)
    r = np.hypot(c.coords[0], c.coords[1])
    c.target_mollifier = 0.25 * (1.0 + np.tanh(4.0 * (r - 4.0))) * (1.0 - np.tanh(4.0 * (r - 9.0)))
    c.initial = _pulses(c, rng, 4, 1e-2, 0.06)
    return c


def _wave(n, steps, save, rng):
    """The cost target covers the control, as above."""
    c = mc.periodic_wave_1d(n=n, nsteps=steps, save_interval=save)
    x = c.coords[0]
    inside = np.nonzero((x >= 0.1) & (x <= 0.9))[0]
    c.target_mollifier = 0.25 * (1.0 + np.tanh(50.0 * (x - 0.2))) * (1.0 - np.tanh(50.0 * (x - 0.8)))
    c.patches = [dataclasses.replace(p, extent=(int(inside[0]) + 1, int(inside[-1]) + 1, 1, -1, 1, -1))
                 if p.type == mc.COST_TARGET else p for p in c.patches]
    c.initial = _pulses(c, rng, 3, 1e-2, 0.04)
    return c


def _flow(n, steps, save, seed):
    """kolmogorov3d's problem with its random solenoidal field made on the GPU."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device="cpu").manual_seed(int(seed) & 0x7FFFFFFF)
    k1 = torch.fft.fftfreq(n, d=1.0 / n, dtype=torch.float64).to(dev)
    kz, ky, kx = k1[:, None, None], k1[None, :, None], k1[None, None, :]
    k2 = kx ** 2 + ky ** 2 + kz ** 2
    safe = torch.where(k2 > 0, k2, torch.ones_like(k2))
    amp = torch.where(k2 > 0, k2 * torch.exp(-k2 / 16.0) / safe.sqrt(), torch.zeros_like(k2))
    # random phases of the modes that carry energy (|k| < 16); the spectrum has died there
    m = min(16, n // 2)
    hat = []
    for _ in range(3):
        noise = torch.randn(2 * m, 2 * m, 2 * m, 2, dtype=torch.float64, generator=g).to(dev)
        full = torch.zeros(n, n, n, dtype=torch.complex128, device=dev)
        idx = (torch.arange(2 * m, device=dev) - m) % n
        full[idx[:, None, None], idx[None, :, None], idx[None, None, :]] = torch.view_as_complex(noise)
        hat.append(full * amp)
    div = (kx * hat[0] + ky * hat[1] + kz * hat[2]) / safe
    u = torch.stack([torch.fft.ifftn(h - k * div).real for h, k in zip(hat, (kx, ky, kz))])
    u = u * (0.05 / (u ** 2).sum(0).mean().sqrt())
    u = u.reshape(3, -1).cpu().numpy()
    x1 = np.arange(n) / n
    coords = np.empty((3, n, n, n))
    coords[0], coords[1], coords[2] = x1, x1[:, None], x1[:, None, None]
    npts = n ** 3
    target = mc.quiescent_state(3, npts)
    q = target.copy()
    q[1:4] = u
    q[4] += 0.5 * (u ** 2).sum(axis=0)
    dt = 0.5 / n / 1.15 / math.sqrt(3.0)
    return mc.Case(
        name="flow%d" % n, nd=3, n=(n, n, n), coords=coords.reshape(3, -1),
        periodicity=(mc.PLANE,) * 3, periodic_length=(1.0, 1.0, 1.0), viscous=True,
        dissipation=False, reynolds=500.0, prandtl=0.7,
        patches=[mc.Patch("forcing", mc.KOLMOGOROV, 0, (1, -1, 1, -1, 1, -1), (4.0, 0.01, 0, 0))],
        target=target, control_mollifier=np.zeros(npts), target_mollifier=np.zeros(npts),
        dt=dt, nsteps=steps, save_interval=save, initial=q)


def _sizes(case):
    """Odd sizes of the ensemble's members, spread over [lo, hi]."""
    m = case["members"]
    r = np.random.Generator(np.random.PCG64(m))
    return [int(2 * r.integers(case["lo"] // 2, case["hi"] // 2 + 1) + 1) for _ in range(m)]


def _problem(case, seed):
    """The mc.Case (a list of them for the ensemble) and the control of a case."""
    rng = np.random.Generator(np.random.PCG64(seed))
    f = case["family"]
    if f == "wave":
        c = _wave(case["n"], case["steps"], case["save"], rng)
        return c, _control(rng, c, 1, 4 * c.nsteps)
    if f in ("monopole", "loop"):
        c = _monopole(case["n"], case["steps"], case.get("save", 8), rng)
        return c, _control(rng, c, case.get("instances", 1), 4 * c.nsteps)
    if f == "shooting":
        c = mc.mixing_layer(nx=case["nx"], ny=case["ny"], seed=int(seed), nsteps=case["steps"],
                            save_interval=case["save"])
        return c, _control(rng, c, 1, 4 * c.nsteps * case["segments"])[0]
    if f == "ensemble":
        cs = [_monopole(n, case["steps"], case["save"], rng) for n in _sizes(case)]
        return cs, [_control(rng, c, 1, 4 * c.nsteps) for c in cs]
    return _flow(case["n"], case["steps"], case["save"], seed), None


def _segments(c, case, seed):
    """Initial conditions of the shooting segments: the layer with another perturbation in
    each (so that the matching conditions are not met), and their start times."""
    rng = np.random.Generator(np.random.PCG64(seed + 1))
    ics = []
    for _ in range(case["segments"]):
        q = _pulses(c, rng, 2, 1e-3, 0.05)
        ics.append(q)
    return ics, [k * c.nsteps * c.dt for k in range(case["segments"])]


def prepare(case, seed):
    from magudi_amd.group import RegionGroup
    from magudi_amd.multishoot import MultipleShooting
    from magudi_amd.solver import Region, Solver
    problem, control = _problem(case, seed)
    f = case["family"]
    state = {"case": case, "control": control}
    if f == "ensemble":
        state["group"] = RegionGroup(problem)
        return state
    if f == "shooting":
        state["shooting"] = MultipleShooting(problem, nsplit=case["segments"], nts=case["steps"],
                                             penalty_weight=1.0, save_interval=case["save"])
        state["ics"], state["t0s"] = _segments(problem, case, seed)
        return state
    r = Region(problem, n_instances=case.get("instances", 1))
    q = problem.initial_state()
    for s in r.states:
        s.initialCondition = q
    if case.get("held", -1) >= 0:
        r.set_step_store(1)
        r.set_window_cache(case["held"])
    state["region"], state["solver"] = r, Solver(r)
    return state


def run(state):
    case, control = state["case"], state["control"]
    f = case["family"]
    if f == "ensemble":
        G = state["group"]
        G.restart()
        return [{"sensitivity": s, "gradient": g, "J": j}
                for s, g, j in G.run_adjoint_merged(controls=control)]
    if f == "shooting":
        M = state["shooting"]
        J = M.msforward(state["ics"], state["t0s"], control=control)
        out = M.msadjoint()
        return {"J": np.array([J]), "ic_grad": out["ic_grad"], "control_grad": out["control_grad"],
                "sensitivity": out["ctrl_ip"], "total": np.array([out["total"]])}
    r, s = state["region"], state["solver"]
    r.restart()
    if f == "loop":
        return _loop(r, s, control)
    if f == "flow":
        if not case["adjoint"]:
            s.runForward()
            return {"state": r.states[0].conservedVariables}
        s.runForwardCheckpointed()
        J = r.terminalKineticEnergy()
        s.runAdjointCheckpointed(terminal=True)
        return {"J": J, "adjoint": r.states[0].adjointVariables}
    if f == "monopole" and not case["adjoint"]:
        J = s.runForward(control=control)
        return {"J": J, "state": [x.conservedVariables for x in r.states]}
    sens, grad, J = s.runAdjoint(control=control)
    return {"sensitivity": sens, "gradient": grad, "J": J,
            "adjoint": r.states[0].adjointVariables}


def _loop(r, s, control):
    from magudi_amd.solver import RK4Integrator
    ti = RK4Integrator()
    J, time = np.zeros(1), 0.0
    for step in range(1, s.nTimesteps + 1):
        for i in (1, 2, 3, 4):
            if i in (2, 4):
                time += 0.5 * s.dt
            ti.substepForward(r, time, s.dt, step, i, control[:, 4 * (step - 1) + i - 1])
            J += ti.norm[i - 1] * s.dt * r.functional()
    return {"J": J, "state": r.states[0].conservedVariables}


def work(case):
    """Bytes: one state in, one out for each stage evaluation and stage update (16 nv 8 B a
    point and forward step, 40 nv 8 B a point and forward + adjoint step), the result
    fields; flops: the operators' multiply-adds and the fluxes."""
    f = case["family"]
    if f == "ensemble":
        pts, nv, adj = sum(n * n for n in _sizes(case)), 4, True
    elif f == "shooting":
        pts, nv, adj = case["nx"] * case["ny"] * case["segments"], 4, True
    elif f == "wave":
        pts, nv, adj = case["n"], 3, True
    elif f == "loop":
        pts, nv, adj = case["n"] ** 2, 4, False
    elif f == "monopole":
        pts, nv, adj = case["n"] ** 2 * case["instances"], 4, case["adjoint"]
    else:
        pts, nv, adj = case["n"] ** 3, 5, case["adjoint"]
    steps = pts * case["steps"]
    flops = {3: 150, 4: 330, 5: 850}[nv]
    return {"bytes": steps * nv * 8.0 * (40 if adj else 16) + pts * nv * 8.0,
            "flops": steps * 4.0 * flops * (3 if adj else 1)}


# ------------------------------------------------------------------- the plain 64-bit model
_H48 = [Fraction(1498139, 5080320), Fraction(1107307, 725760), Fraction(20761, 80640),
        Fraction(1304999, 725760), Fraction(299527, 725760), Fraction(103097, 80640),
        Fraction(670091, 725760), Fraction(5127739, 5080320)]
_C48 = [Fraction(4, 5), Fraction(-1, 5), Fraction(4, 105), Fraction(-1, 280)]


def _closure():
    """The 8 x 12 boundary rows of the SBP 4-8 first derivative: H D is antisymmetric but
    for its corner -1/2, takes the interior stencil where it leaves the block, and is exact
    on polynomials up to degree 4; its three free entries are 541/1000, -27/400, 187/250."""
    known = {(0, 0): Fraction(-1, 2), (5, 6): Fraction(541, 1000), (5, 7): Fraction(-27, 400),
             (6, 7): Fraction(187, 250)}
    for i in range(8):
        for j in range(8, 12):
            if 1 <= j - i <= 4:
                known[i, j] = _C48[j - i - 1]
    unknown = [(i, j) for i in range(8) for j in range(i + 1, 8) if (i, j) not in known]
    col = {ij: k for k, ij in enumerate(unknown)}
    rows = []
    for i in range(8):
        for p in range(5):
            row = [Fraction(0)] * (len(unknown) + 1)
            row[-1] = _H48[i] * (p * Fraction(i) ** (p - 1) if p else 0)
            for j in range(12):
                a, b, s = (i, j, 1) if i <= j else (j, i, -1)
                if i == j and i > 0:
                    continue
                xp = Fraction(j) ** p if p else Fraction(1)
                if (a, b) in col:
                    row[col[a, b]] += s * xp
                elif (a, b) in known:
                    row[-1] -= s * known[a, b] * xp
            rows.append(row)
    m, r = len(unknown), 0
    for c in range(m):                                  # Gauss-Jordan in exact fractions
        k = next(k for k in range(r, len(rows)) if rows[k][c])
        rows[r], rows[k] = rows[k], rows[r]
        rows[r] = [v / rows[r][c] for v in rows[r]]
        for k in range(len(rows)):
            if k != r and rows[k][c]:
                w = rows[k][c]
                rows[k] = [x - w * y for x, y in zip(rows[k], rows[r])]
        r += 1
    q = dict(known)
    q.update({ij: rows[k][-1] for ij, k in col.items()})
    d = np.zeros((8, 12))
    for i in range(8):
        for j in range(12):
            a, b, s = (i, j, 1) if i <= j else (j, i, -1)
            if (a, b) in q:
                d[i, j] = float(s * q[a, b] / _H48[i])
    return d


def _matrices(n, periodic):
    """Dense first derivative, fourth difference, its transpose and the norm weights."""
    D, E = np.zeros((n, n)), np.zeros((n, n))
    i = np.arange(n)
    for k in range(1, 5):
        np.add.at(D, (i, (i + k) % n), float(_C48[k - 1]))
        np.add.at(D, (i, (i - k) % n), -float(_C48[k - 1]))
    for k, c in ((-2, 1.0), (-1, -4.0), (0, 6.0), (1, -4.0), (2, 1.0)):
        np.add.at(E, (i, (i + k) % n), c)
    h = np.ones(n)
    if not periodic:
        B = _closure()
        D[:8], D[-8:] = 0.0, 0.0
        D[:8, :12] = B
        D[-8:, -12:] = -B[::-1, ::-1]
        for m in (0, 1):
            for r, c in ((m, slice(0, 5)), (n - 1 - m, slice(n - 5, n))):
                E[r] = 0.0
                E[r, c] = (1.0, -4.0, 6.0, -4.0, 1.0)
        w = np.array([float(v) for v in _H48])
        h[:8], h[-8:] = w, w[::-1]
    return D, E, E.T.copy(), h


class _Model:
    """The spatial operator of a problem on (instances, components, z, y, x) tensors."""

    def __init__(self, c, dev):
        self.c, self.nd, self.dev = c, c.nd, dev
        T = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)  # noqa: E731
        self.shape = tuple(reversed(c.n[:c.nd]))
        grid = lambda a: T(a).reshape(self.shape)  # noqa: E731
        nd = c.nd
        self.M, self.h, hw = [], [], []
        for d in range(nd):
            D, E, Et, w = _matrices(c.n[d], c.periodicity[d] != mc.NONE)
            x = np.moveaxis(np.asarray(c.coords[d]).reshape(self.shape), nd - 1 - d, -1)
            x = x.reshape(-1, c.n[d])[0]
            if c.periodicity[d] == mc.PLANE:
                L, n = c.periodic_length[d], c.n[d]
                g = np.concatenate([x[-4:] - L, x, x[:4] + L])
                hd = sum(float(_C48[k - 1]) * (g[4 + k:4 + k + n] - g[4 - k:4 - k + n]) for k in range(1, 5))
            else:
                hd = D @ x
            view = [1] * nd
            view[nd - 1 - d] = -1
            self.M.append((T(D), T(E), T(Et)))
            self.h.append(T(hd).reshape(view))
            hw.append(T(w).reshape(view))
        self.hw = hw
        det = torch.ones(self.shape, dtype=torch.float64, device=dev)
        self.H = det.clone()
        for d in range(nd):
            det = det * self.h[d]
            self.H = self.H * hw[d]
        self.jac, self.H = 1.0 / det, self.H * det
        self.metric = []
        for d in range(nd):
            m = torch.ones([1] * nd, dtype=torch.float64, device=dev)
            for e in range(nd):
                if e != d:
                    m = m * self.h[e]
            self.metric.append(m)
        self.target = T(c.target).reshape((nd + 2,) + self.shape)
        self.moll = grid(c.target_mollifier)
        self.cmoll = grid(c.control_mollifier)
        self.pbar = self.prim(self.target[None])[2][0]
        self.cost = self.force = None
        self.act = None
        self.damp = torch.zeros(self.shape, dtype=torch.float64, device=dev)
        self.far = []
        for p in c.patches:
            sl = self._box(p)
            if p.type == mc.COST_TARGET:
                self.cost = torch.zeros(self.shape, dtype=torch.float64, device=dev)
                self.cost[sl] = self.moll[sl] * self.H[sl]
            elif p.type == mc.ACTUATOR:
                self.act = torch.as_tensor(c.patch_points(p), device=dev)
            elif p.type == mc.KOLMOGOROV:
                k = p.params[1] * torch.sin(2 * math.pi * int(p.params[0]) * grid(c.coords[1]))
                self.force = k - (k * self.H).sum() / self.H.sum()
            elif p.type == mc.SPONGE:
                d = abs(p.normal_dir) - 1
                a, b = self._range(p, d)
                arc = self.h[d].reshape(-1).abs()[a:b]
                run = torch.cumsum(arc, 0) - arc
                xi = run / run[-1]
                if p.normal_dir < 0:
                    back = torch.flip(torch.cumsum(torch.flip(arc, (0,)), 0) - torch.flip(arc, (0,)), (0,))
                    xi = back / back[0]
                view = [1] * nd
                view[nd - 1 - d] = -1
                self.damp[sl] += (p.params[0] * (1.0 - xi) ** p.params[1]).reshape(view)
            elif p.type == mc.FAR_FIELD:
                self.far.append((sl, self._incoming(p, sl)))
        self.src = [(s, s.amplitude * torch.exp(-9.0 / (2.0 * s.radius ** 2) * sum(
            (grid(c.coords[d]) - s.location[d]) ** 2 for d in range(nd)))) for s in c.sources]

    def _range(self, p, d):
        a, b = p.extent[2 * d], p.extent[2 * d + 1]
        n = self.c.n[d]
        return (a + n if a < 0 else a - 1), (b + n + 1 if b < 0 else b)

    def _box(self, p):
        return tuple(slice(*self._range(p, d)) for d in reversed(range(self.nd)))

    def _incoming(self, p, sl):
        """sigma J A+(target) of a far-field patch by the spectral projectors of the flux
        Jacobian, whose eigenvalues are u_n and u_n +- c."""
        d, nd, g = abs(p.normal_dir) - 1, self.nd, self.c.gamma
        qt = self.target[(slice(None),) + sl].reshape(nd + 2, -1).T.contiguous()
        def flux(q):
            return self.flux(q.reshape((1, nd + 2) + (1,) * nd), d, None).reshape(-1)
        A = torch.stack([torch.autograd.functional.jacobian(flux, q) for q in qt])
        rho, u, pr, T = self.prim(qt.T.reshape((1, nd + 2, -1)))
        un, cs = u[d][0], torch.sqrt(g * pr[0] / rho[0])
        I = torch.eye(nd + 2, dtype=torch.float64, device=self.dev)
        lam = [un, un + cs, un - cs]
        out = torch.zeros_like(A)
        for k in range(3):
            P = I.expand_as(A)
            for j in range(3):
                if j != k:
                    P = P @ (A - lam[j][:, None, None] * I) / (lam[k] - lam[j])[:, None, None]
            keep = torch.where(p.normal_dir * lam[k] < 0, torch.zeros_like(lam[k]), lam[k])
            out = out + keep[:, None, None] * P
        m = (self.metric[d] * self.jac)[sl].reshape(-1)
        sigma = math.copysign(p.params[0], p.normal_dir) / float(_H48[0])
        return sigma * m[:, None, None] * out

    def apply(self, M, x, d):
        dim = x.dim() - 1 - d
        y = x.transpose(dim, -1).contiguous()
        return (y.reshape(-1, y.shape[-1]) @ M.T).reshape(y.shape).transpose(dim, -1)

    def prim(self, q):
        g, nd = self.c.gamma, self.nd
        rho = q[:, 0]
        u = [q[:, 1 + i] / rho for i in range(nd)]
        p = (g - 1.0) * (q[:, nd + 1] - 0.5 * rho * sum(v * v for v in u))
        return rho, u, p, g * p / ((g - 1.0) * rho)

    def flux(self, q, d, visc):
        rho, u, p, _ = self.prim(q)
        f = [q[:, 1 + d]] + [q[:, 1 + i] * u[d] + (p if i == d else 0.0) for i in range(self.nd)]
        f.append(u[d] * (q[:, self.nd + 1] + p))
        if visc is not None:
            tau, hf = visc
            for i in range(self.nd):
                f[1 + i] = f[1 + i] - tau[i][d]
            f[-1] = f[-1] - sum(u[i] * tau[i][d] for i in range(self.nd)) + hf[d]
        return torch.stack(f, 1)

    def rhs(self, q, time, force):
        c, nd = self.c, self.nd
        visc = None
        if c.viscous:
            _, u, _, T = self.prim(q)
            mu = 1.0 / c.reynolds
            la, ka = (c.bulk_ratio - 2.0 / 3.0) * mu, mu / c.prandtl
            grad = [[self.jac * self.metric[d] * self.apply(self.M[d][0], w, d) for d in range(nd)]
                    for w in u + [T]]
            dil = la * sum(grad[i][i] for i in range(nd))
            tau = [[mu * (grad[i][j] + grad[j][i]) + (dil if i == j else 0.0) for j in range(nd)]
                   for i in range(nd)]
            visc = tau, [-ka * x for x in grad[nd]]
        r = 0.0
        for d in range(nd):
            r = r - self.apply(self.M[d][0], self.metric[d] * self.flux(q, d, visc), d)
        if c.dissipation:
            for d in range(nd):
                t = self.apply(self.M[d][2], -self.metric[d].abs() * self.apply(self.M[d][1], q, d), d)
                r = r + c.dissipation_amount * t / self.hw[d]
        r = r * self.jac
        dq = q - self.target
        r = r - self.damp * dq
        for sl, A in self.far:
            s = (slice(None), slice(None)) + sl
            v = dq[s]
            w = torch.einsum("pij,bjp->bip", A, v.reshape(v.shape[0], nd + 2, -1))
            pad = torch.zeros_like(r)
            pad[s] = w.reshape(v.shape)
            r = r - pad
        add = torch.zeros_like(r)
        for s, shape in self.src:
            add[:, nd + 1] += math.cos(2 * math.pi * s.frequency * time + s.phase) * shape
        if force is not None:
            e = torch.zeros((q.shape[0], self.cmoll.numel()), dtype=torch.float64, device=self.dev)
            e[:, self.act] = force * self.cmoll.reshape(-1)[self.act]
            add[:, nd + 1] += e.reshape(add[:, nd + 1].shape)
        r = r + add
        if self.force is not None:
            k = torch.zeros_like(add)
            k[:, 1] = self.force
            r = r + q[:, :1] * k
        return r

    def sound(self, q):
        """The cost density's quadrature per instance."""
        p = self.prim(q)[2] - self.pbar
        return (p * p * self.cost).flatten(1).sum(1)


_B = (1.0 / 6.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 6.0)


def _forward(m, q, steps, control, keep=False):
    """RK4 steps; J per instance, the final state and the state at the start of each step."""
    dt, time = m.c.dt, 0.0
    J = torch.zeros(q.shape[0], dtype=torch.float64, device=q.device)
    start = []
    with torch.no_grad():
        for s in range(steps):
            if keep:
                start.append(q)
            ys, q = _stages(m, q, time, s, control)
            if m.cost is not None:
                for b, y in zip(_B, ys[1:] + [q]):
                    J += b * dt * m.sound(y)
            time += dt
    return J, q, start


def _stages(m, q, time, s, control):
    dt = m.c.dt
    f = (lambda i: None) if control is None else (lambda i: control[:, 4 * s + i])
    y, ys, acc = q, [], q
    for i, (a, ct) in enumerate(((0.5, 0.0), (0.5, 0.5), (1.0, 0.5), (0.0, 1.0))):
        ys.append(y)
        k = m.rhs(y, time + ct * dt, f(i))
        acc = acc + _B[i] * dt * k
        y = q + a * dt * k
    return ys, acc


def _pull(fn, y, cot):
    """Vector-Jacobian product of fn at y."""
    y = y.detach().requires_grad_(True)
    with torch.enable_grad():
        return torch.autograd.grad(fn(y), y, cot)[0]


def _backward(m, bar, start, control, want_gradient):
    """The adjoint of the RK4 steps from d/dq(T): (sensitivity, gradient, d/dq0)."""
    dt, n = m.c.dt, len(start)
    grad, sens = None, torch.zeros(bar.shape[0], dtype=torch.float64, device=bar.device)
    moll = H = None
    if want_gradient:
        moll, H = m.cmoll.reshape(-1)[m.act], m.H.reshape(-1)[m.act]
        grad = torch.zeros((bar.shape[0], 4 * n, len(m.act)), dtype=torch.float64, device=bar.device)
    for s in reversed(range(n)):
        time = s * dt
        with torch.no_grad():
            ys, qn = _stages(m, start[s], time, s, control)
        if m.cost is not None:
            bar = bar + _B[3] * dt * _pull(lambda y: m.sound(y).sum(), qn, None)
        total, yb = bar, None
        for i in (3, 2, 1, 0):
            kb = _B[i] * dt * bar
            if yb is not None:
                kb = kb + (1.0 if i == 2 else 0.5) * dt * yb
            if want_gradient:
                e = kb[:, m.nd + 1].flatten(1)[:, m.act] / (_B[i] * dt * H) * moll
                grad[:, 4 * s + i] = e
                sens += _B[i] * dt * (e * e * H).sum(1)
            f = None if control is None else control[:, 4 * s + i]
            t = time + (0.0, 0.5, 0.5, 1.0)[i] * dt
            yb = _pull(lambda y: m.rhs(y, t, f), ys[i], kb)
            if m.cost is not None and i > 0:
                yb = yb + _B[i - 1] * dt * _pull(lambda y: m.sound(y).sum(), ys[i], None)
            total = total + yb
        bar = total
    return sens, grad, bar


def _host(x):
    return x.detach().cpu().numpy()


def _exact_seconds(case):
    """A rough estimate of exact()'s time: its operator calls are bound by launches on small
    grids, by memory on large ones."""
    w = work(case)
    adj = case.get("adjoint", case["family"] not in ("loop",))
    calls = case["steps"] * case.get("members", 1) * 4.0 * (4.0 if adj else 1.0)
    return calls * 2e-3 + w["bytes"] * 2e-11


def exact(case, seed):
    f = case["family"]
    if _exact_seconds(case) > 18.0:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    problem, control = _problem(case, seed)
    if f == "ensemble":
        return [_control_run(c, u, 1, dev, False) for c, u in zip(problem, control)]
    if f == "shooting":
        return _shooting_exact(case, problem, control, seed, dev)
    if f == "flow":
        m = _Model(problem, dev)
        q = torch.as_tensor(problem.initial_state(), device=dev).reshape((1, 5) + m.shape)
        _, qT, start = _forward(m, q, case["steps"], None, case["adjoint"])
        if not case["adjoint"]:
            return {"state": _host(qT).reshape(5, -1)}
        ke = lambda y: (0.5 * m.H * (y[:, 1:4] ** 2).sum(1) / y[:, 0]).sum()  # noqa: E731
        _, _, bar = _backward(m, _pull(ke, qT, None), start, None, False)
        return {"J": np.array([float(ke(qT))]), "adjoint": _host(bar / m.H).reshape(5, -1)}
    if f == "loop" or (f == "monopole" and not case["adjoint"]):
        m = _Model(problem, dev)
        y = torch.as_tensor(problem.initial_state(), device=dev).reshape((1, m.nd + 2) + m.shape)
        y = y.expand((len(control),) + y.shape[1:])
        J, qT, _ = _forward(m, y, case["steps"], torch.as_tensor(control, device=dev))
        q = [_host(x).reshape(m.nd + 2, -1) for x in qT]
        return {"J": _host(J), "state": q[0] if f == "loop" else q}
    return _control_run(problem, control, case.get("instances", 1), dev, True)


def _control_run(c, control, instances, dev, want_adjoint):
    m = _Model(c, dev)
    q = torch.as_tensor(c.initial_state(), device=dev).reshape((1, m.nd + 2) + m.shape)
    q = q.expand((instances,) + q.shape[1:])
    u = torch.as_tensor(control, device=dev)
    J, qT, start = _forward(m, q, c.nsteps, u, True)
    sens, grad, bar = _backward(m, torch.zeros_like(qT), start, u, True)
    out = {"sensitivity": _host(sens), "gradient": _host(grad), "J": _host(J)}
    if want_adjoint:
        out["adjoint"] = _host(bar[0] / m.H).reshape(m.nd + 2, -1)
    return out


def _shooting_exact(case, c, control, seed, dev):
    m = _Model(c, dev)
    ics, _ = _segments(c, case, seed)
    S, n = case["segments"], c.nsteps
    u = torch.as_tensor(control.reshape(S, 4 * n, -1), device=dev)
    q = torch.stack([torch.as_tensor(x, device=dev).reshape((m.nd + 2,) + m.shape) for x in ics])
    J, qT, start = _forward(m, q, n, u, True)
    gap = q[1:] - qT[:-1]                    # ic_k - end_(k-1)
    bar = torch.zeros_like(qT)
    bar[:-1] = -gap * m.H
    total = J.sum() + 0.5 * (gap * gap * m.H).sum()
    sens, grad, bar = _backward(m, bar, start, u, True)
    ic = bar / m.H
    ic[1:] += gap
    ip = (ic[1:] ** 2 * m.H).sum()
    return {"J": np.array([float(total)]), "ic_grad": _host(ic).reshape(S, m.nd + 2, -1),
            "control_grad": _host(grad).reshape(S * 4 * n, -1), "sensitivity": _host(sens),
            "total": np.array([float(sens.sum() + ip)])}
