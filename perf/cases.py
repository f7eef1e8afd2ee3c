"""The work that a user of this library has it do, as cases to be timed.

Each case advances a level (or an ensemble, or a differentiated level) by a
few steps of the time loop through the public entry points of ``tenjin_amd``:
``begin_run`` / ``advance``, a captured graph, the host-driven loop of
``compute_dt`` / ``set_dt`` / ``step``, ``GpuBatch`` and ``TangentRun``.  A
pass goes on from the state the last one left, as a run does, unless the case
says otherwise.

``listed()`` gives the cases, ``draw(rng)`` others of the same ranges,
``prepare`` the level with its initial state in device memory, ``run`` one
pass, ``work`` the bytes and operations a pass cannot do without, and
``exact`` the state after the first pass by plain torch in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tenjin_amd as tj
from tenjin_amd import configs, tangent
from tenjin_amd.configs import (ALPHA, ALPHARHO, ALPHARHOEPSILON, ALPHARHOLAMBDA, DEVH, EPSILON, HJ2, LAMBDA, P, RHO,
                                RHO_K, RHO_MIX, RHOU, SOUNDSPEED, TOTAL_E, V_TENSOR, VELOCITY)

PRECS = {"fp64": tj.TJ_PREC_FP64, "mixed": tj.TJ_PREC_MIXED}


def listed():
    return [
        # The smallest: a 1000-cell two-material shock tube, whose steps are
        # replayed as one captured graph of 64 loop bodies.
        {"name": "tube_graph", "kind": "tube", "loop": "graph", "nx": 1000, "box": 1 << 20, "thinc": 0,
         "prec": "fp64", "steps": 64},
        # A small 2D level driven from the host step by step, as the
        # reference's own main loop does (getTimeStep, clamps, advance).
        {"name": "host_loop", "kind": "inclusion", "loop": "host", "nx": 160, "ny": 90, "box": 32, "thinc": 1,
         "prec": "fp64", "steps": 4},
        # The shock/inclusion level at the size of the headline benchmark, in
        # both precisions.
        {"name": "inclusion", "kind": "inclusion", "loop": "device", "nx": 2048, "ny": 1024, "box": 64, "thinc": 1,
         "prec": "fp64", "steps": 4},
        {"name": "inclusion_mixed", "kind": "inclusion", "loop": "device", "nx": 2048, "ny": 1024, "box": 64,
         "thinc": 1, "prec": "mixed", "steps": 4},
        # Odd sizes, MUSCL alone, the state as an AMReX MultiFab holds it (one
        # ghost-grown FAB per box).
        {"name": "inclusion_fabs", "kind": "inclusion", "loop": "fabs", "nx": 701, "ny": 389, "box": 160, "thinc": 0,
         "prec": "fp64", "steps": 4},
        # Axisymmetric underwater explosion with the geometric source.
        {"name": "explosion_rz_mixed", "kind": "explosion", "loop": "device", "nx": 724, "ny": 724, "box": 64,
         "thinc": 1, "prec": "mixed", "steps": 4},
        # A reactive mixture beside air: rootFind in every cell, the burn.  A
        # run from the initial state (the burn of a long run ends in states
        # that the reference refuses).
        {"name": "reactive", "kind": "reactive", "loop": "restart", "nx": 512, "ny": 256, "box": 64, "thinc": 1,
         "prec": "fp64", "steps": 16},
        # An ensemble of independent tubes of uneven size, in one batch.
        {"name": "ensemble_mixed", "kind": "ensemble", "loop": "batch", "n1d": 16, "n2d": 16, "sizes": 6,
         "most1d": 8000, "most2d": 512, "thinc": 1, "prec": "mixed", "steps": 4},
        # Elastoplastic plate impact, in 2D at the size of the differentiated
        # benchmark and in 3D in both precisions, the last one ragged.
        {"name": "plate2d", "kind": "plate", "loop": "device", "dim": 2, "nx": 512, "ny": 512, "nz": 1, "box": 64,
         "prec": "fp64", "steps": 4},
        {"name": "plate3d", "kind": "plate", "loop": "device", "dim": 3, "nx": 144, "ny": 144, "nz": 144, "box": 64,
         "prec": "fp64", "steps": 2},
        {"name": "plate3d_mixed", "kind": "plate", "loop": "device", "dim": 3, "nx": 203, "ny": 160, "nz": 131,
         "box": 64, "prec": "mixed", "steps": 2},
        # Gradient of a probe trace with respect to the six material
        # parameters of a plate impact, two directions per pass group.
        {"name": "gradient", "kind": "gradient", "loop": "tangent", "nx": 160, "ny": 160, "box": 64, "prec": "fp64",
         "steps": 8, "chunk": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tube", "inclusion", "inclusion", "explosion", "reactive", "ensemble", "plate", "plate",
                       "gradient"])
    prec = rng.choice(["fp64", "mixed"])
    box = rng.choice([32, 48, 64, 128])
    if kind == "tube":
        return {"kind": kind, "loop": rng.choice(["graph", "device"]), "nx": _log_int(rng, 200, 16000),
                "box": rng.choice([64, 1 << 20]), "thinc": rng.choice([0, 1]), "prec": prec, "steps": 16}
    if kind == "inclusion":
        nx = _log_int(rng, 64, 2048)
        loop = rng.choice(["device", "device", "graph", "host", "fabs"])
        if loop == "fabs":
            box = max(box, -(-nx // 8))
        return {"kind": kind, "loop": loop, "nx": nx, "ny": max(32, min(1024, int(nx * rng.uniform(0.3, 0.7)))),
                "box": box, "thinc": rng.choice([0, 1, 1]), "prec": prec, "steps": 4}
    if kind == "explosion":
        n = _log_int(rng, 64, 1100)
        return {"kind": kind, "loop": "device", "nx": n, "ny": n, "box": box, "thinc": rng.choice([0, 1]),
                "prec": prec, "steps": 4}
    if kind == "reactive":
        n = _log_int(rng, 64, 900)
        return {"kind": kind, "loop": "restart", "nx": n, "ny": n // 2, "box": box, "thinc": rng.choice([0, 1]),
                "prec": prec, "steps": 16}
    if kind == "ensemble":
        return {"kind": kind, "loop": "batch", "n1d": rng.randint(1, 16), "n2d": rng.randint(1, 16),
                "sizes": rng.randrange(1 << 16), "most1d": 8000, "most2d": rng.choice([128, 256, 512]), "thinc": rng.choice([0, 1]), "prec": prec, "steps": 4}
    if kind == "plate":
        if rng.random() < 0.5:
            n = [_log_int(rng, 48, 900), _log_int(rng, 48, 900), 1]
        else:
            n = [_log_int(rng, 24, 160) for _ in range(3)]
        return {"kind": kind, "loop": "device", "dim": 2 if n[2] == 1 else 3, "nx": n[0], "ny": n[1], "nz": n[2],
                "box": box, "prec": prec, "steps": 2}
    n = _log_int(rng, 40, 200)
    return {"kind": kind, "loop": "tangent", "nx": n, "ny": _log_int(rng, 40, 200), "box": box, "prec": "fp64",
            "steps": 6, "chunk": rng.choice([1, 2, 3])}


# ---------------------------------------------------------------- the levels
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _problem(case, seed):
    """The level of a case (everything but its initial state)."""
    kind, box = case["kind"], case["box"]
    gas = configs.Material.stiffened
    if kind == "tube":
        return configs.Problem("tube", 1, (case["nx"], 1, 1), (1.0, 1.0, 1.0), box, [gas(4.4, 6e8), gas(1.4)],
                               THINC=case["thinc"])
    if kind == "inclusion":
        return configs.Problem("inclusion", 2, (case["nx"], case["ny"], 1), (2.0, 1.0, 1.0), box,
                               [gas(1.4), gas(1.67)], THINC=case["thinc"], bc_lo=(0, 1, 0), bc_hi=(0, 1, 0))
    if kind == "explosion":
        return configs.Problem("explosion", 2, (case["nx"], case["ny"], 1), (1.0, 1.0, 1.0), box,
                               [gas(4.4, 6e8), gas(1.4)], THINC=case["thinc"], RADIAL=1, bc_lo=(1, 0, 0))
    if kind == "reactive":
        mix = configs.Material.mixture_mg(configs.EXPLOSIVE_REACTANT, configs.EXPLOSIVE_PRODUCTS)
        return configs.Problem("reactive", 2, (case["nx"], case["ny"], 1), (1.0, 0.5, 1.0), box, [mix, gas(1.4)],
                               THINC=case["thinc"], REACTIVE=1, bc_lo=(0, 1, 0), bc_hi=(0, 1, 0))
    mats = [configs.Material.usup_solid(**configs.COPPER), configs.Material.usup_solid(**configs.ALUMINIUM)]
    dim = case.get("dim", 2)
    n = (case["nx"], case["ny"], case.get("nz", 1))
    h = 25.6e-3 / 256
    return configs.Problem("plate", dim, n, (h * n[0], h * n[1], h * n[2]), box, mats, SOLID=1, PLASTIC=1,
                           shift_pressure=1)


def _initial(case, pb, seed):
    """The initial primitives [ncomp][nz][ny][nx] of a case, on the device."""
    dev = _device()
    rs = np.random.RandomState(seed % (1 << 31))
    L, kind = pb.layout, case["kind"]
    nz, ny, nx = pb.shape
    U = torch.zeros((L.ncomp, nz, ny, nx), dtype=torch.float64, device=dev)

    def centres(a, n):
        return (torch.arange(n, dtype=torch.float64, device=dev) + 0.5) * (pb.L[a] / n)

    X = centres(0, nx).view(1, 1, nx).expand(nz, ny, nx)
    Y = centres(1, ny).view(1, ny, 1).expand(nz, ny, nx)

    def pick(mask, a, b):
        t = [torch.as_tensor(v, dtype=torch.float64, device=dev) for v in (a, b)]
        return torch.where(mask, t[0], t[1])

    def fill(first, rho0, rho1, u, p):
        a0 = pick(first, 1.0 - configs.ABSENT_ALPHA, configs.ABSENT_ALPHA)
        U[L.comp(ALPHA, 0)] = a0
        U[L.comp(ALPHA, 1)] = 1.0 - a0
        U[L.comp(RHO_K, 0)] = rho0
        U[L.comp(RHO_K, 1)] = rho1
        for r in range(3):
            U[L.comp(VELOCITY, 0, r)] = u[r]
        U[L.comp(P)] = p

    if kind == "tube":  # water-like fluid at high pressure beside air
        left = X < 0.7
        fill(left, 1000.0, 50.0, (0.0, 0.0, 0.0), pick(left, 1e9 * rs.uniform(0.8, 1.2), 1e5))
    elif kind == "inclusion":  # Mach 1.22 shock, light inclusion with a perturbed boundary
        amp, phase = rs.uniform(-0.01, 0.01, 8), rs.uniform(0.0, 2.0 * math.pi, 8)
        th = torch.atan2(Y - 0.5, X - 0.8)
        r = 0.2 * (1.0 + sum(float(amp[k]) * torch.cos((k + 1) * th + float(phase[k])) for k in range(8)))
        outside = torch.hypot(Y - 0.5, X - 0.8) >= r
        rho2, u2, p2 = configs.rankine_hugoniot(1.4, 1.0, 1e5, 1.22)
        shocked = X < 0.5
        fill(outside, pick(shocked, rho2, 1.0), 0.138, (pick(shocked, u2, 0.0), 0.0, 0.0), pick(shocked, p2, 1e5))
    elif kind == "explosion":  # high-pressure gas bubble on the axis, in water
        water = torch.hypot(X, Y - 0.5) >= 0.2 * rs.uniform(0.9, 1.1)
        fill(water, 1000.0, 1270.0, (0.0, 0.0, 0.0), pick(water, 1e5, 8.29e8))
    elif kind == "reactive":  # ignition region, unburnt explosive, air beyond a wavy line
        edge = 0.6 + 0.02 * torch.sin(2.0 * math.pi * (4.0 * Y + rs.uniform()))
        ignition = X < 0.1
        fill(X < edge, 1000.0, 1.2, (0.0, 0.0, 0.0), pick(ignition, 2e9, 1e5))
        noise = torch.from_numpy(rs.random_sample((nz, ny, nx))).to(dev)
        U[L.comp(LAMBDA)] = torch.where(ignition, torch.full_like(noise, 0.2), 0.5 + 0.5 * noise)
        U[L.comp(RHO_MIX, 0, 0)] = U[L.comp(RHO_K, 0)]
        U[L.comp(RHO_MIX, 0, 1)] = U[L.comp(RHO_K, 0)]
    else:  # plate, gradient: copper flyer on aluminium, interface tilted by 5 degrees
        t = math.radians(5.0)
        copper = (X - 0.5 * pb.L[0]) * math.cos(t) + (Y - 0.5 * pb.L[1]) * math.sin(t) < 0.0
        fac = 1.0 + 1e-3 * (2.0 * torch.from_numpy(rs.random_sample((nz, ny, nx))).to(dev) - 1.0)
        fill(copper, configs.COPPER["rho0"] * fac, configs.ALUMINIUM["rho0"] * fac,
             (pick(copper, rs.uniform(200.0, 600.0), 0.0), 0.0, 0.0), 0.0)
        for r in range(3):
            U[L.comp(V_TENSOR, 0, r, r)] = 1.0
    return U


def _sizes(case):
    """Cells of the 1D problems and sides of the 2D ones: the case's own."""
    rs = np.random.RandomState(case["sizes"])
    return ([int(rs.randint(500, case["most1d"] + 1)) for _ in range(case["n1d"])],
            [int(rs.randint(64, case["most2d"] + 1)) for _ in range(case["n2d"])])


def _ensemble(case, seed):
    """Its problems: materials, ratios and interface from the seed."""
    out = []
    for dim, sizes in enumerate(_sizes(case), 1):
        for q, n in enumerate(sizes):
            out += configs.ensemble(seed=(seed + 1009 * len(out)) % (1 << 31), n1d=dim == 1, n2d=dim == 2,
                                    n1d_range=(n, n), side_range=(n, n), thinc=case["thinc"])
    return out


def _probe(pb):
    """u_x two cells into the target, where the impact arrives at once."""
    nz, ny, nx = pb.shape
    return pb.layout.comp(VELOCITY, 0, 0), nx // 2 + 2, ny // 2, 0


def prepare(case, seed):
    prec, loop = PRECS[case["prec"]], case["loop"]
    if loop == "batch":
        batch = tj.GpuBatch(_ensemble(case, seed))
        batch.init_from_prims()
        batch.begin_run()
        return {"batch": batch, "prec": prec, "steps": case["steps"]}
    pb = _problem(case, seed)
    prims = _initial(case, pb, seed)
    if loop == "tangent":
        pb.prims = prims.cpu().numpy()
        run_ = tangent.TangentRun(pb, tangent.ALL_DIRECTIONS, chunk=case["chunk"])
        return {"tangent": run_, "steps": case["steps"], "probe": _probe(pb)}
    if loop == "fabs":
        level = tj.GpuFabLevel(pb, ghost_fill=0.0)
        level.init_from_prims(prims.cpu().numpy(), pb.shift_pressure)
    else:
        level = tj.GpuLevel(pb)
        level.init_from_device(prims, pb.shift_pressure)
    state = {"level": level, "prec": prec, "steps": case["steps"], "loop": loop, "n": 0}
    if loop == "restart":
        state["prims"] = prims
    if loop != "host":
        level.begin_run()
    if loop == "graph":
        level.graph_capture(case["steps"], prec)
    level.sync()
    return state


def run(state):
    if "batch" in state:
        state["batch"].advance(state["steps"], state["prec"])
        return list(state["batch"].S)
    if "tangent" in state:
        t = state["tangent"]
        trace, _ = t.run(state["steps"], state["probe"])
        return {"value": trace[:, 0], "derivative": trace[:, 1:], "state": t.g.S}
    g = state["level"]
    if state["loop"] == "graph":
        g.graph_launch()
    elif state["loop"] == "host":
        for _ in range(state["steps"]):
            dt = g.compute_dt()
            if state["n"] < 5:
                dt *= 0.2
            g.set_dt(dt)
            g.step(state["prec"])
            state["n"] += 1
    else:
        if state["loop"] == "restart":
            g.init_from_device(state["prims"], g.pb.shift_pressure)
            g.begin_run()
        g.advance(state["steps"], state["prec"])
    return list(g.fabS) if state["loop"] == "fabs" else g.S


# ---------------------------------------------------------------- the least work
def work(case):
    """Bytes: per cell and step each RK stage reads its primitives and the
    rest of the state once and writes the new state once (3 state arrays and
    2 times the conserved variables, FP64).  Operations: the formulas' own
    additions, products, quotients and roots, each counted once."""
    kind, steps = case["kind"], case["steps"]
    if kind == "ensemble":
        one, two = _sizes(case)
        c1, c2 = sum(one), sum(n * n for n in two)
        return {"bytes": 464.0 * steps * (c1 + c2), "flops": steps * (740.0 * c1 + 1330.0 * c2)}
    cells = case["nx"] * case.get("ny", 1) * case.get("nz", 1)
    dim = 1 if kind == "tube" else case.get("dim", 2)
    if kind in ("plate", "gradient"):
        per_b, per_f = 952.0, 2.0 * (dim * 1190.0 + 230.0) + 1000.0
        if kind == "gradient":  # values once, then each direction's derivative state and twice the operations
            per_b, per_f = per_b * 7.0, per_f * 13.0
    elif kind == "reactive":  # some 30 trial pressures in each of 3 root findings
        per_b, per_f = 576.0, 2.0 * (dim * 340.0 + 50.0) + 3.0 * 30.0 * 20.0 + 150.0
    else:
        per_b, per_f = 464.0, 2.0 * (dim * 293.0 + 40.0) + 74.0
    return {"bytes": per_b * cells * steps, "flops": per_f * cells * steps}


# ---------------------------------------------------------------- the exact state
def _exact_level(pb, prims, steps):
    return (_Solid if pb.SOLID else _Fluid)(pb, prims).advance(steps)


def exact(case, seed):
    if case["loop"] == "batch":
        out = []
        for pb in _ensemble(case, seed):
            prims = torch.from_numpy(pb.prims).to(_device())
            out.append(_exact_level(pb, prims, case["steps"]).state())
        return out
    pb = _problem(case, seed)
    level = _exact_level(pb, _initial(case, pb, seed), case["steps"])
    S = level.state()
    if case["loop"] == "tangent":
        c, i, j, k = _probe(pb)
        values = [float(s[c, k, j, i]) for s in level.history]
        # the derivatives of the non-smooth step have no plain form to take them from
        return {"value": np.array(values), "derivative": None, "state": S}
    if case["loop"] == "fabs":
        out = []
        cuts = [_boxes(pb.n[a], pb.max_grid_size) if a < pb.dim else [(0, 0)] for a in range(3)]
        for z in cuts[2]:
            for y in cuts[1]:
                for x in cuts[0]:
                    g = [2 if a < pb.dim else 0 for a in range(3)]
                    fab = torch.zeros([S.shape[0]] + [b[1] - b[0] + 1 + 2 * g[a] for a, b in ((2, z), (1, y), (0, x))],
                                      dtype=torch.float64, device=S.device)
                    fab[:, g[2]:fab.shape[1] - g[2], g[1]:fab.shape[2] - g[1], g[0]:fab.shape[3] - g[0]] = \
                        S[:, z[0]:z[1] + 1, y[0]:y[1] + 1, x[0]:x[1] + 1]
                    out.append(fab)
        return out
    return S


def _boxes(n, most):
    """BoxArray::maxSize along one dimension: (low, high) of each box."""
    if n <= most:
        return [(0, n - 1)]
    ratio, bs, nlen = 1, most, n
    while bs % 2 == 0 and nlen % 2 == 0:
        ratio, bs, nlen = ratio * 2, bs // 2, nlen // 2
    blocks = -(-nlen // bs)
    size, extra = divmod(nlen, blocks)
    out, hi = [], n - 1
    for b in range(blocks - 1):
        width = (size + 1 if b < extra else size) * ratio
        out.append((hi - width + 1, hi))
        hi -= width
    return sorted(out + [(0, hi)])


def _near(x, axis, by):
    """x at the neighbour cell `by` = +-1 along an axis, the edge cell repeated."""
    n = x.shape[axis]
    if by > 0:
        return torch.cat([x.narrow(axis, 1, n - 1), x.narrow(axis, n - 1, 1)], axis)
    return torch.cat([x.narrow(axis, 0, 1), x.narrow(axis, 0, n - 1)], axis)


def _slope(m, c, p):
    """MUSCL with van Leer's limiter: the cell's low and high face values."""
    r = (c - m) / (p - c)
    r = torch.where(torch.isfinite(r), r, torch.zeros_like(r))
    phi = torch.where(r > 0, torch.minimum(2.0 * r, torch.full_like(r, 2.0)) / (1.0 + r), torch.zeros_like(r))
    half = 0.5 * (phi * 0.5 * (p - m))
    return c - half, c + half


def _unit(a):
    """cleanUpAlpha of volume fractions without NaN."""
    a = [torch.where(x < 0, torch.full_like(x, 1e-6), torch.clamp(x, max=1.0)) for x in a]
    total = sum(a)
    return [x * (1.0 / total) for x in a]


class _Level:
    """The time loop on one level, with the state as a dict of lists of
    [nz][ny][nx] tensors by variable."""

    def __init__(self, pb, prims):
        self.pb, self.dev, self.dim = pb, prims.device, pb.dim
        self.start = prims.clone()
        self.M, self.mats = pb.nmat, pb.materials
        self.dx = pb.dx()
        self.history, self.n = [], 0
        self.gg = [m.gamma - 1.0 for m in self.mats]

    def get(self, var, count):
        return [self.start[self.pb.layout.start[var] + q].clone() for q in range(count)]

    def put(self, S, var, parts):
        for q, x in enumerate(parts):
            S[self.pb.layout.start[var] + q] = x

    def advance(self, steps):
        for _ in range(steps):
            speeds = [self.dx[d] / (self.s["a"] + self.s["u"][d].abs()) for d in range(self.dim)]
            dt = self.pb.CFL * min(float(x.min()) for x in speeds) * (0.2 if self.n < 5 else 1.0)
            self.step(dt)
            self.n += 1
            if self.pb.SOLID:
                self.history.append(self.state())
        return self

    def faces(self, L, R, d, fields):
        """Left and right states of the faces along d: the neighbours' face
        values, and at the domain's ends the edge cell's own, mirrored where
        the boundary reflects."""
        axis, n = -1 - d, self.pb.n[d]
        left, right = {}, {}
        for key in fields:
            left[key], right[key] = [], []
            for q in range(len(R[key])):
                lo, hi = R[key][q].narrow(axis, 0, 1), L[key][q].narrow(axis, n - 1, 1)
                if key == "u" and q == d:
                    lo, hi = (-lo if self.pb.bc_lo[d] else lo), (-hi if self.pb.bc_hi[d] else hi)
                left[key].append(torch.cat([lo, R[key][q]], axis))
                right[key].append(torch.cat([L[key][q], hi], axis))
        return left, right

    def jump(self, F, d):
        """F at the low face minus F at the high face of each cell."""
        n = self.pb.n[d]
        return F.narrow(-1 - d, 0, n) - F.narrow(-1 - d, 1, n)

    def neighbours(self, x, d, odd=False):
        m, p = _near(x, -1 - d, -1), _near(x, -1 - d, 1)
        n = self.pb.n[d]
        if odd and self.pb.bc_lo[d]:
            m.narrow(-1 - d, 0, 1).neg_()
        if odd and self.pb.bc_hi[d]:
            p.narrow(-1 - d, n - 1, 1).neg_()
        return m, p

    def reconstruct(self, s, d, fields):
        L, R = {}, {}
        for key in fields:
            L[key], R[key] = [], []
            for q, x in enumerate(s[key]):
                m, p = self.neighbours(x, d, key == "u" and q == d)
                lo, hi = _slope(m, x, p)
                L[key].append(lo)
                R[key].append(hi)
        return L, R


class _Fluid(_Level):
    """Stiffened gases and Mie-Gruneisen fluids, MUSCL (+ THINC/BVD) and HLLC;
    with a mixture material also its mass fraction and phase densities."""

    def __init__(self, pb, prims):
        super().__init__(pb, prims)
        self.mix = next((m for m, t in enumerate(self.mats) if t.mixture), -1)
        s = {"al": self.get(ALPHA, 2), "rk": self.get(RHO_K, 2), "u": self.get(VELOCITY, 3), "p": self.get(P, 1)}
        if self.mix >= 0:
            s["lam"] = self.get(LAMBDA, 1)
        self.conserved(s)
        s["p"], s["a"] = s["p"][0], s["a"][0]
        self.s = s
        zero = torch.zeros(pb.shape, dtype=torch.float64, device=self.dev)
        # what THINC's selection reads of earlier passes: the last THINC value
        # of each cell's high face, the last pass' star-state alphas, and those
        # of the last pass in the same direction
        self.thr = [zero.clone() for _ in range(2)]
        self.star = [zero.clone() for _ in range(2)]
        self.edge_star = {}
        self.edges = {}
        for d in range(self.dim):
            lo, hi = torch.zeros(pb.n[d], dtype=torch.bool), torch.zeros(pb.n[d], dtype=torch.bool)
            for b in _boxes(pb.n[d], pb.max_grid_size):
                lo[b[0]], hi[b[1]] = True, True
            shape = [1, 1, 1]
            shape[2 - d] = pb.n[d]
            self.edges[d] = (lo.view(shape).to(self.dev), hi.view(shape).to(self.dev))

    # closures -----------------------------------------------------------
    def mix_gamma(self, lam):
        t = self.mats[self.mix]
        return (lam * t.gamma * t.CV + (1 - lam) * t.gamma2 * t.CV2) / (lam * t.CV + (1 - lam) * t.CV2) - 1.0

    def sums(self, al, ar, lam=None, rk=None, ra=None, rb=None):
        G = Ent = Pnt = 0.0
        for m, t in enumerate(self.mats):
            if m == self.mix:
                g1, g2 = t.gamma - 1.0, t.gamma2 - 1.0
                G = G + al[m] / self.mix_gamma(lam)
                Ent = Ent + (lam * (t.eref * ar[m]) + (1 - lam) * (t.eref2 * ar[m]))
                Pnt = Pnt + (t.pref * al[m] / g1) * lam * rk / ra + (t.pref2 * al[m] / g2) * (1 - lam) * rk / rb
            else:
                G, Ent, Pnt = G + al[m] / self.gg[m], Ent + t.eref * ar[m], Pnt + t.pref * al[m] / self.gg[m]
        return G, Ent, Pnt

    def sound(self, al, ar, rk, rho, p, lam=None, ra=None, rb=None):
        a = xt = 0.0
        for m, t in enumerate(self.mats):
            if m == self.mix:
                g1, g2, r = t.gamma - 1.0, t.gamma2 - 1.0, rk[m]
                de = lam * ((t.pref - p) / (g1 * r * r)) + (1 - lam) * ((t.pref2 - p) / (g2 * r * r))
                c2 = (p / (r * r) - de) / (lam / (ra * g1) + (1 - lam) / (rb * g2))
                xi = 1.0 / self.mix_gamma(lam)
            else:
                c2, xi = p * (self.gg[m] + 1.0) / rk[m] - t.pref / rk[m], 1.0 / self.gg[m]
            a = a + torch.clamp(xi * c2 * ar[m] / rho, min=0.0)
            xt = xt + xi * al[m]
        a = torch.where(a <= 0, torch.full_like(a, 1e-6), a)
        return torch.sqrt(a / xt)

    def conserved(self, s):
        """Conserved variables and sound speed of primitives (in place)."""
        p = s["p"][0]
        s["ar"] = [a * r for a, r in zip(s["al"], s["rk"])]
        s["rho"] = [sum(s["ar"])]
        rho, more = s["rho"][0], {}
        if self.mix >= 0:
            t, lam, rk = self.mats[self.mix], s["lam"][0], s["rk"][self.mix]
            s["arl"] = [lam * s["al"][self.mix] * rk]
            ra = rk * (lam + (1 - lam) * ((p - t.pref) / (p - t.pref2)) *
                       ((t.CV2 * (t.gamma2 - 1.0)) / (t.CV * (t.gamma - 1.0))))
            rb = (1 - lam) / (1.0 / rk - lam / ra)
            s["rmix"] = [ra, rb]
            more = {"lam": lam, "ra": ra, "rb": rb}
        ke = sum(0.5 * rho * u * u for u in s["u"])
        G, Ent, Pnt = self.sums(s["al"], s["ar"], rk=s["rk"][self.mix], **more)
        s["E"] = [p * G + Ent - Pnt + ke]
        s["ru"] = [u * rho for u in s["u"]]
        s["a"] = [self.sound(s["al"], s["ar"], s["rk"], rho, p, **more)]

    def root(self, s, ke, lam, rk):
        """Phase densities of the mixture in thermal equilibrium, by bisection
        on the reactants' density to a relative width of 1e-7."""
        t = self.mats[self.mix]
        g1, g2 = t.gamma - 1.0, t.gamma2 - 1.0

        def other(ra):
            return (1 - lam) / (1.0 / rk - lam / ra)

        def f(ra):
            rb = other(ra)
            G, Ent, Pnt = self.sums(s["al"], s["ar"], lam, rk, ra, rb)
            p = (s["E"] - ke - Ent + Pnt) / G
            return (p - t.pref) / (ra * g1 * t.CV) - (p - t.pref2) / (rb * g2 * t.CV2)

        lo, hi = lam * rk + 1e-10, torch.full_like(rk, 1e6)
        first, last = f(lo), f(hi)
        ra = 0.5 * (lo + hi)
        open_ = torch.ones_like(rk, dtype=torch.bool)
        for test, at in ((first.abs() <= 1e-4, lo.clone()), (last.abs() <= 1e-4, hi.clone())):
            ra = torch.where(open_ & test, at, ra)
            open_ &= ~test
        for _ in range(100):
            same = torch.sign(f(ra)) == torch.sign(first)
            lo, hi = torch.where(open_ & same, ra, lo), torch.where(open_ & ~same, ra, hi)
            ra = torch.where(open_, 0.5 * (lo + hi), ra)
            open_ = open_ & ~((lo - hi).abs() / (lo + hi) < 1e-7)
            if not bool(open_.any()):
                break
        ends = (lam > 1.0 - 1e-3) | (lam < 1e-3)
        return torch.where(ends, rk, ra), torch.where(ends, rk, other(ra))

    def primitive(self, s):
        s["rk"] = [r / a for r, a in zip(s["ar"], s["al"])]
        rho = s["rho"] = sum(s["ar"])
        s["u"] = [r / rho for r in s["ru"]]
        ke = sum(0.5 * rho * u * u for u in s["u"])
        more = {}
        if self.mix >= 0:
            lam, rk = s["arl"] / s["ar"][self.mix], s["rk"][self.mix]
            ra, rb = self.root(s, ke, lam, rk)
            s["lam"], s["rmix"] = [lam], [ra, rb]
            more = {"lam": lam, "rk": rk, "ra": ra, "rb": rb}
        G, Ent, Pnt = self.sums(s["al"], s["ar"], **more)
        s["p"] = (s["E"] - ke - Ent + Pnt) / G

    # one directional pass --------------------------------------------------
    def thinc(self, s, d, L, R):
        axis, pb = -1 - d, self.pb
        lo_edge, hi_edge = self.edges[d]
        yn = [-1.0 / (8.0 * self.dx[q]) for q in range(2)]
        ula, ura, thl, thr, mixed = [], [], [], [], []
        for m in range(2):
            a = s["al"][m]
            aL, aR = _near(a, axis, -1), _near(a, axis, 1)
            mn = torch.minimum(aL, aR)
            mx = torch.maximum(aL, aR) - mn
            theta = torch.sign(aR - aL)
            C = torch.where(mx < 1e-20, torch.zeros_like(a), (a - mn + 1e-20) / (mx + 1e-20))
            mixed.append((C > 1e-4) & (C < 0.999999 - 1e-4) & ((aR - a) * (a - aL) >= 0))
            nv = torch.ones_like(a)
            if self.dim == 2:
                W, E = _near(a, -1, -1), _near(a, -1, 1)
                N, S_, NE, NW = _near(a, -2, 1), _near(a, -2, -1), _near(E, -2, 1), _near(W, -2, 1)
                SE, SW = _near(E, -2, -1), _near(W, -2, -1)
                gx = yn[0] * (NE + 2 * E + SE - NW - 2 * W - SW)
                gy = yn[1] * (NE + 2 * N + NW - SW - 2 * S_ - SE)
                norm = torch.sqrt(gx * gx + gy * gy)
                nv = torch.where(norm < 1e-20, torch.zeros_like(a), ((gx, gy)[d] / norm).abs())
            beta = nv * pb.THINCbeta + 0.01
            ch, th = torch.cosh(beta), torch.tanh(beta)
            A = (torch.exp(theta * beta * (2 * C - 1)) / ch - 1) / th
            thr.append(mn + mx / 2 * (1 + theta * ((th + A) / (1 + A * th))))
            thl.append(mn + mx / 2 * (1 + theta * A))
            ula.append(L["al"][m])
            ura.append(R["al"][m])
        for m in range(2):
            flag = mixed[-1]
            a = s["al"][m]
            prev, nxt = (lambda x: _near(x, axis, -1)), (lambda x: _near(x, axis, 1))
            edge = self.edge_star.get(d)
            edge = torch.zeros_like(a) if edge is None else edge[m].narrow(axis, 1, pb.n[d])
            own_l = torch.where(mixed[m], thl[m], self.star[m])
            own_r = torch.where(mixed[m], thr[m], self.thr[m])
            URl = torch.where(lo_edge, prev(a), prev(ura[m]))
            TRl = torch.where(lo_edge, torch.zeros_like(a), torch.where(prev(mixed[m]), prev(thr[m]), prev(self.thr[m])))
            ULr = torch.where(hi_edge, nxt(a), nxt(ula[m]))
            TLr = torch.where(hi_edge, edge, torch.where(nxt(mixed[m]), nxt(thl[m]), nxt(self.star[m])))

            def variation(pl, pr):
                one = (URl - pl).abs() + (pr - ULr).abs()
                two = (TRl - pl).abs() + (pr - TLr).abs()
                three = (URl - pl).abs() + (pr - TLr).abs()
                four = (TRl - pl).abs() + (pr - ULr).abs()
                return torch.minimum(torch.minimum(one, two), torch.minimum(three, four))

            take = flag & (variation(own_l, own_r) < variation(ula[m], ura[m]))
            L["al"][m] = torch.where(take, own_l, ula[m])
            R["al"][m] = torch.where(take, own_r, ura[m])
        L["al"], R["al"] = _unit(L["al"]), _unit(R["al"])
        self.thr = [torch.where(mixed[m], thr[m], self.thr[m]) for m in range(2)]

    def fluxes(self, s, d):
        prims = ["al", "rk", "u", "p"] + (["lam"] if self.mix >= 0 else [])
        t = {k: (s[k] if isinstance(s[k], list) else [s[k]]) for k in prims}
        L, R = self.reconstruct(t, d, prims)
        if self.pb.THINC:
            self.thinc(s, d, L, R)
        self.conserved(L)
        self.conserved(R)
        keys = ["al", "ar", "rho", "u", "E", "p", "a"] + (["arl"] if self.mix >= 0 else [])
        l, r = self.faces(L, R, d, keys)
        rho_l, rho_r, ul, ur = l["rho"][0], r["rho"][0], l["u"][d], r["u"][d]
        SR = torch.maximum(ul.abs() + l["a"][0], ur.abs() + r["a"][0])
        SL = -SR
        Ss = (r["p"][0] - l["p"][0] + ul * rho_l * (SL - ul) - ur * rho_r * (SR - ur)) / \
             (rho_l * (SL - ul) - rho_r * (SR - ur))
        use_left = (SL >= 0) | (Ss >= 0)
        star = ~(SL >= 0) & ((Ss >= 0) | (SR >= 0))

        def side(key, q=0):
            return torch.where(use_left, l[key][q], r[key][q])

        rho, u, E, p = side("rho"), [side("u", q) for q in range(3)], side("E"), side("p")
        SK = torch.where(use_left, SL, SR)
        mult = torch.where(((Ss - u[d]) / Ss).abs() < 1e-20, torch.ones_like(Ss), (SK - u[d]) / (SK - Ss))

        def added(f, us, uk):
            return torch.where(star, f + SK * (us - uk), f)

        F = {"S": Ss}
        ar = [side("ar", m) for m in range(2)]
        al = [side("al", m) for m in range(2)]
        ru = [x * rho for x in u]
        ru_s = [mult * rho * Ss if q == d else mult * ru[q] for q in range(3)]
        u_s = ru_s[d] / sum(mult * x for x in ar)
        F["al"] = [x * u_s for x in al]
        F["ar"] = [added(x * u[d], mult * x, x) for x in ar]
        F["ru"] = [added(ru[q] * u[d] + (p if q == d else 0.0), ru_s[q], ru[q]) for q in range(3)]
        E_s = mult * rho * (E / rho + (Ss - u[d]) * (Ss + p / (rho * (SK - u[d]))))
        F["E"] = added(E * u[d] + u[d] * p, E_s, E)
        if self.mix >= 0:
            x = side("arl")
            F["arl"] = added(x * u[d], mult * x, x)
        self.star = [x.narrow(-1 - d, 0, self.pb.n[d]) for x in al]
        self.edge_star[d] = al
        return F

    def stage(self, s, dt):
        new = {"al": list(s["al"]), "ar": list(s["ar"]), "ru": list(s["ru"]), "E": s["E"]}
        if self.mix >= 0:
            new["arl"] = s["arl"]
        for d in range(self.dim):
            F, r = self.fluxes(s, d), dt / self.dx[d]
            for m in range(2):
                new["al"][m] = new["al"][m] + r * (self.jump(F["al"][m], d) - s["al"][m] * self.jump(F["S"], d))
                new["ar"][m] = new["ar"][m] + r * self.jump(F["ar"][m], d)
            for q in range(3):
                new["ru"][q] = new["ru"][q] + r * self.jump(F["ru"][q], d)
            new["E"] = new["E"] + r * self.jump(F["E"], d)
            if self.mix >= 0:
                new["arl"] = new["arl"] + r * self.jump(F["arl"], d)
        self.primitive(new)
        return new

    def step(self, dt):
        s = self.s
        for k in ("E", "rho", "arl"):
            if isinstance(s.get(k), list):
                s[k] = s[k][0]
        new = self.stage(self.stage(s, dt), dt)
        for k, v in new.items():
            new[k] = [0.5 * a + 0.5 * b for a, b in zip(s[k], v)] if isinstance(v, list) else 0.5 * s[k] + 0.5 * v
        if self.pb.REACTIVE and self.mix >= 0:
            al, ar, y0, p = new["al"][self.mix], new["ar"][self.mix], new["arl"], new["p"]

            def burn(y):
                z = y - dt * (20.0 * ar ** 0.5 * y ** 0.5 * (p / 1e6) ** 1.2)
                return torch.where(al < 0.5, y, torch.clamp(z, min=0.0))

            new["arl"] = 0.5 * y0 + 0.5 * burn(burn(y0))
            self.primitive(new)
        if self.pb.RADIAL:
            i = torch.arange(self.pb.n[0], dtype=torch.float64, device=self.dev)
            f = dt * ((-2.0 if self.dim == 1 else -1.0) / ((i + 0.5) * self.dx[0]))
            u, p = new["u"], new["p"]
            new["E"] = new["E"] + f * (new["E"] * u[0] + u[0] * p)
            new["ar"] = [x + f * (x * u[0]) for x in new["ar"]]
            ru = new["ru"]
            new["ru"] = [ru[0] + f * (ru[0] * u[0]), ru[1] + f * (ru[1] * u[0]), ru[2]]
            self.primitive(new)
        new["al"] = _unit(new["al"])
        more = {}
        if self.mix >= 0:
            more = {"lam": new["lam"][0], "ra": new["rmix"][0], "rb": new["rmix"][1]}
        new["a"] = self.sound(new["al"], new["ar"], new["rk"], new["rho"], new["p"], **more)
        self.s = new

    def state(self):
        S, s = self.start.clone(), self.s
        for var, key in ((ALPHA, "al"), (ALPHARHO, "ar"), (RHO_K, "rk"), (RHO, "rho"), (RHOU, "ru"), (VELOCITY, "u"),
                         (TOTAL_E, "E"), (P, "p"), (SOUNDSPEED, "a"), (LAMBDA, "lam"), (ALPHARHOLAMBDA, "arl"),
                         (RHO_MIX, "rmix")):
            if key in s:
                self.put(S, var, s[key] if isinstance(s[key], list) else [s[key]])
        return S


class _Solid(_Level):
    """Us-up solids with perfect plasticity: MUSCL, the 5-wave flux, the
    radial return and the clean-up of the inverse deformation V (a list of
    nine, row by row)."""

    def __init__(self, pb, prims):
        super().__init__(pb, prims)
        s = {"al": self.get(ALPHA, 2), "rk": self.get(RHO_K, 2), "u": self.get(VELOCITY, 3), "p": self.get(P, 1),
             "V": self.get(V_TENSOR, 9), "e": self.get(EPSILON, 2)}
        ar = [a * r for a, r in zip(s["al"], s["rk"])]
        G, _, Pnt = self.sums(s["al"], ar, s["rk"], self.start[pb.layout.start[HJ2]])
        s["p"] = [s["p"][0] + Pnt / G]
        self.conserved(s, 0)
        self.devh, _ = self.strain(s["V"])
        self.s = {k: (v[0] if k in ("rho", "E", "p", "a", "hj2") else v) for k, v in s.items()}

    # closures ---------------------------------------------------------------
    @staticmethod
    def mul_t(A, B):
        return [sum(A[3 * r + k] * B[3 * c + k] for k in range(3)) for r in range(3) for c in range(3)]

    @staticmethod
    def mul(A, B):
        return [sum(A[3 * r + k] * B[3 * k + c] for k in range(3)) for r in range(3) for c in range(3)]

    @staticmethod
    def det(M):
        return M[0] * (M[4] * M[8] - M[5] * M[7]) - M[1] * (M[3] * M[8] - M[5] * M[6]) + \
            M[2] * (M[3] * M[7] - M[4] * M[6])

    @classmethod
    def inverse(cls, M):
        D = cls.det(M)
        adj = [M[4] * M[8] - M[5] * M[7], M[2] * M[7] - M[1] * M[8], M[1] * M[5] - M[2] * M[4],
               M[5] * M[6] - M[3] * M[8], M[0] * M[8] - M[2] * M[6], M[2] * M[3] - M[0] * M[5],
               M[3] * M[7] - M[4] * M[6], M[1] * M[6] - M[0] * M[7], M[0] * M[4] - M[1] * M[3]]
        return [x / D for x in adj]

    def strain(self, V):
        """Deviatoric Hencky strain of V and its second invariant."""
        G = self.mul_t(V, V)
        H = [0.25 * (a - b) for a, b in zip(G, self.inverse(G))]
        return H, sum(x * x for x in H)

    def hugoniot(self, t, rho):
        """p_H, e_H and their density derivatives."""
        eta, de = 1.0 - t.rho0 / rho, t.rho0 / (rho * rho)
        den, k = 1.0 - t.s * eta, t.rho0 * t.c0 * t.c0
        p = k * eta / (den * den)
        dp = k * (1.0 + t.s * eta) / (den * den * den) * de
        return p, p * eta / (2.0 * t.rho0), dp, (dp * eta + p * de) / (2.0 * t.rho0)

    def sums(self, al, ar, rk, hj2):
        G = Ent = Pnt = 0.0
        for m, t in enumerate(self.mats):
            p, e, _, _ = self.hugoniot(t, rk[m])
            G = G + al[m] / self.gg[m]
            Ent = Ent + (ar[m] * e + al[m] * (t.G0 * hj2))
            Pnt = Pnt + al[m] / self.gg[m] * (p - t.G0 * hj2)
        return G, Ent, Pnt

    def sound(self, al, ar, rk, rho, p, hj2):
        a = xt = 0.0
        for m, t in enumerate(self.mats):
            g = self.gg[m]
            ph, _, dp, de = self.hugoniot(t, rk[m])
            c2 = (p * (g + 1.0) - ph + (g + 1.0) * t.G0 * hj2) / rk[m] + dp - g * rk[m] * de + 4.0 / 3.0 * t.G0 / rk[m]
            a = a + torch.clamp(1.0 / g * c2 * ar[m] / rho, min=0.0)
            xt = xt + 1.0 / g * al[m]
        a = torch.where(a <= 0, torch.full_like(a, 1e-6), a)
        return torch.sqrt(a / xt)

    def shear(self, al):
        up = sum(t.G0 * (al[m] / self.gg[m]) for m, t in enumerate(self.mats))
        return up / sum(al[m] / self.gg[m] for m in range(2))

    def conserved(self, s, d):
        p = s["p"][0]
        s["ar"] = [a * r for a, r in zip(s["al"], s["rk"])]
        rho = sum(s["ar"])
        s["rho"] = [rho]
        s["are"] = [e * r for e, r in zip(s["e"], s["ar"])]
        H, hj2 = self.strain(s["V"])
        ke = sum(0.5 * rho * u * u for u in s["u"])
        G, Ent, Pnt = self.sums(s["al"], s["ar"], s["rk"], hj2)
        s["E"] = [p * G + Ent - Pnt + ke]
        s["ru"] = [u * rho for u in s["u"]]
        Gs = self.shear(s["al"])
        s["sig"] = [(-p if r == d else 0.0) + 2.0 * Gs * H[3 * r + d] for r in range(3)]
        s["a"] = [self.sound(s["al"], s["ar"], s["rk"], rho, p, hj2)]
        s["hj2"] = [hj2]

    def primitive(self, s):
        s["rk"] = [r / a for r, a in zip(s["ar"], s["al"])]
        s["e"] = [e / r for e, r in zip(s["are"], s["ar"])]
        rho = s["rho"] = sum(s["ar"])
        _, s["hj2"] = self.strain(s["V"])
        s["u"] = [r / rho for r in s["ru"]]
        ke = sum(0.5 * rho * u * u for u in s["u"])
        G, Ent, Pnt = self.sums(s["al"], s["ar"], s["rk"], s["hj2"])
        s["p"] = (s["E"] - ke - Ent + Pnt) / G

    # one directional pass ---------------------------------------------------
    def fluxes(self, s, d):
        prims = ["al", "rk", "u", "p", "V", "e"]
        L, R = self.reconstruct({k: (s[k] if isinstance(s[k], list) else [s[k]]) for k in prims}, d, prims)
        self.conserved(L, d)
        self.conserved(R, d)
        l, r = self.faces(L, R, d, ["al", "ar", "are", "rho", "u", "E", "a", "sig", "V"])
        for t in (l, r):
            t["ru"] = [u * t["rho"][0] for u in t["u"]]
        SR = torch.maximum(l["u"][d].abs() + l["a"][0], r["u"][d].abs() + r["a"][0])
        SL = -SR
        ml, mr = l["rho"][0] * (SL - l["u"][d]), r["rho"][0] * (SR - r["u"][d])
        Ss = (l["sig"][d] - r["sig"][d] + l["ru"][d] * (SL - l["u"][d]) - r["ru"][d] * (SR - r["u"][d])) / (ml - mr)

        def star(K, SK):
            mult = torch.where(((Ss - K["u"][d]) / Ss).abs() < 1e-20, torch.ones_like(Ss),
                               (SK - K["u"][d]) / (SK - Ss))
            rho = K["rho"][0]
            T = {"al": K["al"], "ar": [mult * x for x in K["ar"]], "are": [mult * x for x in K["are"]]}
            T["rho"] = sum(T["ar"])
            T["ru"] = [mult * rho * Ss if q == d else mult * K["ru"][q] for q in range(3)]
            T["u"] = [x / T["rho"] for x in T["ru"]]
            T["V"] = [K["V"][q] if q // 3 == d else mult * K["V"][q] for q in range(9)]
            T["E"] = mult * rho * (K["E"][0] / rho + (Ss - K["u"][d]) *
                                   (Ss - K["sig"][d] / (rho * (SK - K["u"][d]))))
            rk = [a / b for a, b in zip(T["ar"], T["al"])]
            b = sum(T["al"][m] / self.gg[m] * t.G0 / rk[m] for m, t in enumerate(self.mats))
            b = torch.where(b > 0, b, torch.zeros_like(b))
            T["ct"] = torch.nan_to_num(torch.sqrt(b / sum(T["al"][m] / self.gg[m] for m in range(2))), nan=0.0)
            return T

        ls, rs = star(l, SL), star(r, SR)
        SLT, SRT = Ss - ls["ct"], Ss + rs["ct"]
        left = (SL >= 0) | (Ss >= 0)
        only_k = (SL >= 0) | (~left & ~(SR >= 0))
        both = ~only_k & torch.where(left, ~(SLT >= 0), SRT >= 0)

        def side(a, b):
            return torch.where(left, a, b)

        SK, SKT = side(SL, SR), side(SLT, SRT)
        u, sig = [side(l["u"][q], r["u"][q]) for q in range(3)], [side(l["sig"][q], r["sig"][q]) for q in range(3)]
        V, E = [side(l["V"][q], r["V"][q]) for q in range(9)], side(l["E"][0], r["E"][0])
        Vs, us = [side(ls["V"][q], rs["V"][q]) for q in range(9)], [side(ls["u"][q], rs["u"][q]) for q in range(3)]
        rus, Es, rho_s = [side(ls["ru"][q], rs["ru"][q]) for q in range(3)], side(ls["E"], rs["E"]), side(ls["rho"], rs["rho"])
        jl, jr = ls["rho"] * (Ss - SLT), rs["rho"] * (Ss - SRT)
        sig_s = [(jl * jr * (l["u"][q] - r["u"][q]) + jl * r["sig"][q] - jr * l["sig"][q]) / (jl - jr) for q in range(3)]
        dS = Ss - SKT
        ru2, E2, V2 = list(rus), Es, list(Vs)
        for q in range(3):
            if q == d:
                continue
            ru2[q] = rus[q] + (sig_s[q] - sig[q]) / dS
            uq = ru2[q] / rho_s
            E2 = E2 + (uq * sig_s[q] - u[q] * sig[q]) / dS
            for c in range(3):
                V2[3 * q + c] = Vs[3 * q + c] + Vs[3 * d + c] * (uq - u[q]) / dS

        def total(f, k, ks, kss=None):
            one = f + SK * (ks - k)
            two = one if kss is None else torch.where(both, one + SKT * (kss - ks), one)
            return torch.where(only_k, f, two)

        F = {"S": Ss, "al": [side(ls["al"][m], rs["al"][m]) * us[d] for m in range(2)]}
        for key in ("ar", "are"):
            k = [side(l[key][m], r[key][m]) for m in range(2)]
            F[key] = [total(k[m] * u[d], k[m], side(ls[key][m], rs[key][m])) for m in range(2)]
        ru = [side(l["ru"][q], r["ru"][q]) for q in range(3)]
        F["ru"] = [total(ru[q] * u[d] - sig[q], ru[q], rus[q], ru2[q]) for q in range(3)]
        F["E"] = total(E * u[d] - sum(u[q] * sig[q] for q in range(3)), E, Es, E2)
        F["V"] = [total(V[3 * q + c] * u[d] - V[3 * d + c] * u[q], V[3 * q + c], Vs[3 * q + c], V2[3 * q + c])
                  for q in range(3) for c in range(3)]
        F["Vd"] = [torch.where(only_k, V[3 * d + c], Vs[3 * d + c]) for c in range(3)]
        return F

    def stage(self, s, dt):
        new = {k: (list(s[k]) if isinstance(s[k], list) else s[k]) for k in ("al", "ar", "are", "ru", "E", "V")}
        for d in range(self.dim):
            F, r = self.fluxes(s, d), dt / self.dx[d]
            jS = self.jump(F["S"], d)
            for m in range(2):
                new["al"][m] = new["al"][m] + r * (self.jump(F["al"][m], d) - s["al"][m] * jS)
                for key in ("ar", "are"):
                    new[key][m] = new[key][m] + r * self.jump(F[key][m], d)
            for q in range(3):
                new["ru"][q] = new["ru"][q] + r * self.jump(F["ru"][q], d)
            new["E"] = new["E"] + r * self.jump(F["E"], d)
            for q in range(9):
                new["V"][q] = new["V"][q] + r * (self.jump(F["V"][q], d) - 2.0 / 3.0 * s["V"][q] * jS +
                                                 s["u"][q // 3] * self.jump(F["Vd"][q % 3], d))
        self.primitive(new)
        return new

    def plastic(self, s):
        """Radial return to the yield surface; V takes the Cayley form of the
        scaled strain in every cell."""
        H, hj2 = self.strain(s["V"])
        J = torch.sqrt(hj2)
        JT = JB = norm = 0.0
        for m, t in enumerate(self.mats):
            Jn = torch.where(t.G0 * J * math.sqrt(3.0) > t.yield_stress,
                             torch.full_like(J, t.yield_stress / (math.sqrt(3.0) * t.G0)), J)
            s["e"][m] = s["e"][m] + math.sqrt(2.0 / 3.0) * (J - Jn)
            s["are"][m] = s["e"][m] * s["ar"][m]
            w = s["al"][m] / self.gg[m]
            JB, JT, norm = JB + w * J, JT + w * Jn, norm + w
        JB, JT = JB / norm, JT / norm
        rest = (JB == 0) & (JT == 0)
        ratio = torch.where(rest, torch.ones_like(JB), JT / torch.where(rest, torch.ones_like(JB), JB))
        eye = [1.0 if q % 4 == 0 else 0.0 for q in range(9)]
        half = [0.5 * h * ratio for h in H]
        s["V"] = self.mul(self.inverse([e - h for e, h in zip(eye, half)]), [e + h for e, h in zip(eye, half)])

    def unimodular(self, s):
        """V <- the symmetric square root of V V^T scaled to determinant 1
        (the root by Denman and Beavers' iteration)."""
        Y = self.mul_t(s["V"], s["V"])
        Z = [torch.full_like(Y[0], 1.0 if q % 4 == 0 else 0.0) for q in range(9)]
        for _ in range(12):
            Yi, Zi = self.inverse(Y), self.inverse(Z)
            Y, Z = [0.5 * (a + b) for a, b in zip(Y, Zi)], [0.5 * (a + b) for a, b in zip(Z, Yi)]
        scale = self.det(Y) ** (-1.0 / 3.0)
        total = sum(s["al"])
        s["V"] = [y * scale * total / total for y in Y]

    def step(self, dt):
        s = self.s
        new = self.stage(self.stage(s, dt), dt)
        for k, v in new.items():
            new[k] = [0.5 * a + 0.5 * b for a, b in zip(s[k], v)] if isinstance(v, list) else 0.5 * s[k] + 0.5 * v
        self.plastic(new)
        self.primitive(new)
        self.unimodular(new)
        new["al"] = _unit(new["al"])
        new["a"] = self.sound(new["al"], new["ar"], new["rk"], new["rho"], new["p"], new["hj2"])
        self.s = new

    def state(self):
        S, s = self.start.clone(), self.s
        for var, key in ((ALPHA, "al"), (ALPHARHO, "ar"), (RHO_K, "rk"), (RHO, "rho"), (RHOU, "ru"), (VELOCITY, "u"),
                         (TOTAL_E, "E"), (P, "p"), (SOUNDSPEED, "a"), (V_TENSOR, "V"), (HJ2, "hj2"), (EPSILON, "e"),
                         (ALPHARHOEPSILON, "are")):
            self.put(S, var, s[key] if isinstance(s[key], list) else [s[key]])
        self.put(S, DEVH, self.devh)
        return S
