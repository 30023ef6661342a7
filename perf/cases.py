"""The work that users of this package have it do, as timed cases.

A case is one call (or one recorded interval) of a program that indents tetrahedral cells: a single
``Simulation`` in its different laws, contacts, scatters and sizes; a population of cells in the
inner loop of a fit (reset to new physics, whole indentation, curves); and the curve surrogate's
network.  Cells are balls of a cubic lattice, each cube cut into six tetra, nodes jittered by
``+-10 %`` of the spacing and ordered along a Morton curve: about six tetra per node, as the
Delaunay cells of ``nofluidx3d_amd.mesh`` have, but quick enough to make for every state.  A cell of ``m``
lattice spacings in radius has about ``25 (m + 0.5)^3`` tetra.

A state starts in mid-indentation: a smooth displacement of a few per cent strain with a dent under
the indenter, made from the seed, and the indenter in contact.  ``exact`` repeats every run in float64
with plain torch operations.
"""

import functools
import itertools
import math

import numpy as np
import torch

E_SIM = 0.01  # Young's modulus in simulation units (all cells)
CONTACT = 0.1  # penalty constant of substrate and indenter
XI = 0.005  # velocity damping
OUT = "/tmp/nfx_perf_cases/"
SIZES = (6, 512, 512, 512, 512, 256)  # the surrogate's layers


# ---- cases -------------------------------------------------------------------------------------
def listed():
    return [
        # One time step of the smallest cell, called step by step from Python with user code in
        # between: nothing but the cost of a call and its launches.
        {"name": "tiny_step", "kind": "cell", "m": 5, "law": "nh", "indenter": "sphere", "scatter": "tiled", "tile_k": 128,
         "steps": 1, "hist": False, "record": False, "stress": False, "radius_um": 4.0},
        # The small benchmark cell: 100 steps, then the row of recorded quantities (time, indentation,
        # force), which is what its run loop does 200 times.
        {"name": "small_record", "kind": "cell", "m": 10, "law": "nh", "indenter": "sphere", "scatter": "tiled",
         "tile_k": 128, "steps": 100, "hist": False, "record": True, "stress": False, "radius_um": 8.0},
        # A middle-sized Mooney-Rivlin cell under a flat punch, 1000 steps with the indenter force of
        # every step kept (a force curve at full resolution).
        {"name": "mid_hist", "kind": "cell", "m": 16, "law": "mr", "indenter": "plane", "scatter": "tiled", "tile_k": 256,
         "steps": 1000, "hist": True, "record": False, "stress": False, "radius_um": 8.0},
        # Power-law viscoplastic flow with hardening (every tetra flows, the strain is read) up to a
        # frame that shows the von Mises stress and the pressure.
        {"name": "mid_flow_stress", "kind": "cell", "m": 27, "law": "vp_hard", "indenter": "sphere", "scatter": "tiled",
         "tile_k": 256, "steps": 50, "hist": False, "record": False, "stress": True, "radius_um": 9.0},
        # The large benchmark cell (0.46 M nodes, 2.65 M tetra): Mooney-Rivlin with Maxwell flow above a
        # yield stress, contact developed, 200 steps of its protocol.
        {"name": "large_yield", "kind": "cell", "m": 47, "law": "vp_yield", "indenter": "sphere", "scatter": "tiled",
         "tile_k": 256, "steps": 200, "hist": False, "record": False, "stress": False, "radius_um": 10.0},
        # A legacy law with stress outputs on the CSR gather, the deterministic scatter for meshes that
        # tiles do not fit.
        {"name": "legacy_csr", "kind": "cell", "m": 20, "law": "nh2", "indenter": "sphere", "scatter": "csr", "tile_k": 512,
         "steps": 40, "hist": False, "record": False, "stress": True, "radius_um": 8.0},
        # A law that the fused step does not carry (Prony series): plugin by plugin, as third-party plugins run.
        {"name": "plugin_prony", "kind": "cell", "m": 13, "law": "prony", "indenter": "sphere", "scatter": "tiled",
         "tile_k": 512, "steps": 10, "hist": False, "record": False, "stress": False, "radius_um": 8.0},
        # The inner loop of a fit and of the surrogate's data generation: new physics on the same
        # meshes, the whole indentation, the normalised curves.  Uneven cells with Maxwell flow.
        {"name": "batch_flow", "kind": "batch", "cells": 32, "m_lo": 7, "m_hi": 16, "viscous": True, "steps": 600,
         "ncurve": 256},
        # The same for a handful of small elastic cells.
        {"name": "batch_elastic", "kind": "batch", "cells": 6, "m_lo": 5, "m_hi": 9, "viscous": False, "steps": 500,
         "ncurve": 256},
        # The surrogate's answer to the candidates of a few fits, from host features to host curves.
        {"name": "mlp_predict", "kind": "mlp", "rows": 1000, "call": "predict"},
        # The network alone on device-resident features, at the chunk that large candidate sets run in.
        {"name": "mlp_forward", "kind": "mlp", "rows": 65536, "call": "forward"},
        # One Adam step of the surrogate's training at its batch of 4096.
        {"name": "mlp_train", "kind": "mlp", "rows": 4096, "call": "train"},
    ]


def draw(rng):
    """One more case of the same ranges: cells of 3 k to 2.6 M tetra in every law and option, populations
    of 2 to 32 cells, networks of 128 to 65 536 rows."""
    between = lambda lo, hi: lo * (hi / lo) ** rng.random()  # noqa: E731
    kind = rng.choice(["cell", "cell", "cell", "batch", "mlp"])
    if kind == "batch":
        lo = rng.randint(5, 9)
        return {"kind": kind, "cells": round(between(2, 32)), "m_lo": lo, "m_hi": lo + rng.randint(0, 7),
                "viscous": rng.random() < 0.7, "steps": rng.randrange(150, 600), "ncurve": rng.choice([64, 100, 256])}
    if kind == "mlp":
        call = rng.choice(["predict", "forward", "train"])
        rows = round(between(100, 20000)) if call == "predict" else 128 * round(between(1, 512 if call == "forward" else 32))
        return {"kind": kind, "rows": rows, "call": call}
    m = int(between(5, 47.9))
    law = rng.choice(["nh", "mr", "svk", "nh2", "vp_yield", "vp_hard", "prony"])
    scatter = rng.choice(["tiled", "tiled", "tiled", "csr"])
    per_pass = 1 if rng.random() < 0.2 else int(between(2, 600 if m < 20 else 120))
    fused = law != "prony"
    return {"kind": kind, "m": m if fused else min(m, 20), "law": law, "indenter": rng.choice(["sphere", "plane"]),
            "scatter": scatter, "tile_k": 128 if m < 12 else 256, "steps": per_pass if fused else min(per_pass, 20),
            "hist": fused and rng.random() < 0.3, "record": rng.random() < 0.3,
            "stress": law in ("nh2", "vp_yield", "vp_hard", "prony") and rng.random() < 0.3,
            "radius_um": round(rng.uniform(4.0, 10.0), 2)}


# ---- meshes ------------------------------------------------------------------------------------
def _interleave(p):
    key = np.zeros(len(p), np.int64)
    for axis in range(3):
        for bit in range(8):
            key |= ((p[:, axis] >> bit) & 1) << (3 * bit + axis)
    return key


@functools.lru_cache(maxsize=64)
def _ball(m, jitter_seed):
    """(points (N, 3) float64 in lattice spacings, tetra (T, 4)) of a ball whose +x pole, node 1, lies at
    distance m from its centre, node 0; positively oriented."""
    r = m + 1
    n = 2 * r + 1
    g = np.arange(-r, r + 1)
    inside = (g[:, None, None] ** 2 + g[None, :, None] ** 2 + g[None, None, :] ** 2) <= r * r
    whole = np.ones((n - 1, n - 1, n - 1), bool)
    for d in itertools.product((0, 1), repeat=3):
        whole &= inside[d[0]:n - 1 + d[0], d[1]:n - 1 + d[1], d[2]:n - 1 + d[2]]
    cubes = np.argwhere(whole)
    cubes = cubes[np.argsort(_interleave(cubes), kind="stable")]
    step = np.array([n * n, n, 1])
    paths = []
    for p in itertools.permutations(range(3)):  # the six corner-to-corner paths of a cube
        at = [0, step[p[0]], step[p[0]] + step[p[1]], step.sum()]
        even = p in ((0, 1, 2), (1, 2, 0), (2, 0, 1))
        paths.append(at if even else [at[0], at[2], at[1], at[3]])
    tets = ((cubes @ step)[:, None, None] + np.array(paths)[None]).reshape(-1, 4)
    used = np.zeros(n ** 3, bool)
    used[tets.ravel()] = True
    ids = np.flatnonzero(used)
    P = np.stack(np.unravel_index(ids, (n, n, n)), 1)
    key = _interleave(P)
    P = P - r
    key[(P == 0).all(1)] = -2
    key[(P == [m, 0, 0]).all(1)] = -1
    order = np.argsort(key, kind="stable")
    renumber = np.zeros(n ** 3, np.int64)
    renumber[ids[order]] = np.arange(len(ids))
    P = P[order].astype(np.float64)
    P[2:] += np.random.default_rng(jitter_seed).uniform(-0.1, 0.1, (len(P) - 2, 3))
    return P, renumber[tets]


@functools.lru_cache(maxsize=2)
def _grid(m):
    from nofluidx3d_amd.util import vtk

    return vtk.from_tetra(*_ball(m, 1))


# ---- one cell ----------------------------------------------------------------------------------
def _cell_config(c):
    """The reference-format configuration: simulation units with RadiusSIM = m (one length per lattice spacing),
    mass scaling to 1e-5 s per step, the indenter moving all the time at RadiusSIM / 80 000 per step."""
    m, T0 = c["m"], 1e-5
    R = c["radius_um"] * 1e-6
    mr = c["law"] in ("mr", "vp_yield")
    E, nu = (1168.83, 0.46104) if mr else (1000.0, 0.45)
    L0, p0 = R / m, E / E_SIM
    cell = {"RadiusSI": R, "RadiusSIM": float(m), "YoungsModulusSI": E, "PoissonRatio": nu, "InitVTK": "",
            "MooneyRivlinRatio": 0.75 if mr else 1.0,
            "model": {"mr": "MOONEY_RIVLIN", "svk": "SAINT_VENANT_KIRCHHOFF"}.get(c["law"], "NEO_HOOKEAN")}
    if c["law"] == "vp_yield":
        cell |= {"ViscositySI": 100.0, "YieldStressSI": 200.0}
    elif c["law"] == "vp_hard":
        cell |= {"ViscoplasticFlowExponent": 2.0, "HardeningThreshhold": 0.05, "HardeningExponent": 0.3,
                 "ViscoplasticTimeConstantSI": 2.5e-8}
    elif c["law"] == "nh2":
        cell["SecondOrderNeoHookeanFactor"] = 0.4
    elif c["law"] == "prony":
        cell |= {"ViscoelasticWeights": [0.3, 0.2], "ViscoelasticRelaxationTimes": [50.0, 400.0]}
    return {"gpu": 0, "RhoSI": p0 * (T0 / L0) ** 2, "SimulationTimeSI": 1.0, "VTKFramesTotal": 100, "OutputDir": OUT,
            "InitialDistance": 0.0, "MoveTimeSI": 0.2, "VelocitySI": R / 0.8, "SphereRadiusSI": 0.4 * R, "CELL": cell}


START = {"sphere": 9600, "plane": 2400}  # the step a state starts at: indentation 0.12 or 0.03 RadiusSIM


def _start_positions(c, seed):
    """Positions at the start, in simulation units as FP32 values, and the reference positions."""
    P, _ = _ball(c["m"], 1)
    R = float(c["m"])
    X = (P * (R / abs(P[1, 0]))).astype(np.float32).astype(np.float64)
    rng = np.random.default_rng([seed, c["m"]])
    u = np.zeros_like(X)
    for _ in range(4):  # long waves, about 1 % strain each
        k = rng.normal(size=3) * (1.5 / R)
        u += 0.01 / np.linalg.norm(k) * rng.normal(size=3) * np.sin(X @ k + rng.uniform(0, 2 * np.pi))[:, None]
    u *= np.maximum(1 - (X[:, 1:2] / R) ** 2, 0)  # at rest at the two poles in contact
    depth = START[c["indenter"]] / 80000 * R - 0.1 - 0.1 * rng.random()  # the indenter overlaps by 0.1 to 0.2 lengths
    u[:, 1] -= depth * np.exp(-((X[:, 0] ** 2 + X[:, 2] ** 2 + (X[:, 1] - R) ** 2) / (2 * (0.3 * R) ** 2)))
    return (X + u).astype(np.float32).astype(np.float64), X


def _prepare_cell(c, seed):
    from nofluidx3d_amd.Simulation import Simulation

    sim = Simulation(_cell_config(c), scatter=c["scatter"], mesh=_grid(c["m"]), verbose=False, tile_k=c["tile_k"])
    sim.setInteractionSubstrate()
    sim.setInteractionSphere() if c["indenter"] == "sphere" else sim.setInteractionPlane()
    if c["law"] in ("nh", "mr", "svk"):
        sim.setInteractionTetra()
    elif c["law"] == "nh2":
        sim.setInteractionSecondOrderNeoHookean()
    elif c["law"] == "prony":
        sim.setInteractionLinearViscoelastic()
    else:
        sim.setInteractionFiniteStrainViscoplastic()
    law = sim.interactions[-1]
    sim.setInteractionVelocityVerlet()
    if c["stress"]:
        law.write_stress = True
    x, _ = _start_positions(c, seed)
    sim.points.arrayC[...] = x.T.reshape(-1)
    sim.points.writeToGPU()
    sim.time = START[c["indenter"]]
    sim.plan()  # the step's description and tables, which a program builds once
    hist = torch.zeros(c["steps"], dtype=torch.float64, device=sim.device) if c["hist"] else None
    torch.cuda.synchronize()
    return {"c": c, "sim": sim, "law": law, "hist": hist}


# The velocity and the last force of a node are the net of nearly balanced corner forces: over a long run FP32
# rounding grows to 1e-5 .. 1e-4 of them (against float64), which says nothing.  They come back after few steps.
FEW = 20


def _run_cell(s):
    c, sim, law = s["c"], s["sim"], s["law"]
    if c["steps"] == 1 and s["hist"] is None:
        sim.timeStep()
    else:
        sim.advance(c["steps"], tip_hist=s["hist"])
    vv = sim.interactions[-1]
    fused = c["law"] != "prony"
    out = {"x": sim.displacement if fused else sim.points.buf}
    if c["steps"] <= FEW:
        out["v"], out["f"] = vv.velocityB, vv.forceOldB
    if s["hist"] is not None:
        out["hist"] = s["hist"].float()  # the state is FP32: so is a kept curve
    if c["record"]:
        out["row"] = np.array([q() for q in sim.recordedQuantities], np.float32)[1:]
    if c["stress"]:
        out["stress"], out["pressure"] = sim.vonMises.buf, sim.pressure.buf
    if c["law"] in ("vp_yield", "vp_hard"):
        out["plastic"], out["strain"] = law.plasticDeviationB, law.accumulatedStrainB
    elif c["law"] == "prony":
        out["transient"] = law.transientStressB
    return out


# ---- populations -------------------------------------------------------------------------------
def _population(c, seed):
    """Cells of the case (meshes fixed by the case) with physics from the seed, in the ranges the surrogate's
    training data are drawn from; dicts of plain numbers."""
    mesh = np.random.default_rng([c["cells"], c["m_lo"], c["m_hi"]])
    rng = np.random.default_rng([seed, c["cells"]])
    out = []
    for i in range(c["cells"]):
        m, R = int(mesh.integers(c["m_lo"], c["m_hi"] + 1)), float(mesh.uniform(4.0, 10.0))
        while True:
            d = {"m": m, "R": R, "E": 10 ** rng.uniform(2.0, 4.0), "nu": rng.uniform(0.3, 0.49),
                 "eta": 10 ** rng.uniform(0.0, 3.0), "tip": rng.uniform(1.0, 5.0), "speed": 10 ** rng.uniform(-0.3, 1.7),
                 "seed": i}
            d["T0"] = 0.3 * R / d["speed"] / c["steps"]
            if not c["viscous"] or d["E"] / (2 * (1 + d["nu"])) * d["T0"] / d["eta"] <= 0.1:
                break
        out.append(d)
    return out


def _specs(c, seed):
    from nofluidx3d_amd.batch import CellSpec

    return [CellSpec(d["R"], d["R"] / d["m"], d["seed"], d["E"], d["nu"], d["eta"] if c["viscous"] else None, d["tip"],
                     d["speed"]) for d in _population(c, seed)]


def _prepare_batch(c, seed):
    from nofluidx3d_amd.autotune import group_tetra
    from nofluidx3d_amd.batch import CellGroups

    specs = _specs(c, seed)
    meshes = []
    for d in _population(c, seed):
        P, T = _ball(d["m"], d["seed"] % 4)
        meshes.append((P * (d["R"] / d["m"]), T))
    cells = CellGroups(specs, meshes, max_tetra=group_tetra(), steps=c["steps"], ncurve=c["ncurve"])
    return {"c": c, "cells": cells, "specs": specs}


def _run_batch(s):
    cells = s["cells"]
    cells.reset(s["specs"])
    cells.advance(cells.steps)
    curves = cells.curves_normalized().astype(np.float32)  # as the training data keep them
    return {"curves": curves, "x": [g.x for g in cells.groups]}


# ---- the network -------------------------------------------------------------------------------
def _network_inputs(c, seed):
    rng = np.random.default_rng([seed, c["rows"]])
    X = rng.normal(size=(c["rows"], SIZES[0])).astype(np.float32)
    T = rng.normal(size=(c["rows"], SIZES[-1])).astype(np.float32) if c["call"] == "train" else None
    w = rng.uniform(0.3, 2.0, c["rows"]).astype(np.float32) if c["call"] == "train" else None
    return X, T, w


ADAM_STEP = 200  # a training step in mid-training: moments of the gradients' size


def _moments(shape, seed, dev):
    g = torch.Generator().manual_seed(seed)
    m = 2e-5 * torch.randn(shape, generator=g)
    return m.to(dev), (1e-9 + m * m + 2e-10 * torch.rand(shape, generator=g)).to(dev)


def _prepare_mlp(c, seed):
    from nofluidx3d_amd.surrogate.mlp import MLP

    net = MLP(SIZES, seed=seed % 1000)
    X, T, w = _network_inputs(c, seed)
    s = {"c": c, "net": net, "X": X}
    if c["call"] == "predict":
        return s
    net.set_input(X, train=c["call"] == "train")
    if c["call"] == "train":
        s["T"], s["w"] = torch.from_numpy(T).to(net.dev), torch.from_numpy(w).to(net.dev)
        for l in range(net.nl):
            net.mW[l], net.vW[l] = _moments(tuple(net.W[l].shape), 10 * seed + l, net.dev)
            net.mW[l][:, net.sizes[l]:] = 0
            net.mb[l], net.vb[l] = _moments(tuple(net.b[l].shape), 10 * seed + 5 + l, net.dev)
        net.step = ADAM_STEP
    torch.cuda.synchronize()
    return s


def _run_mlp(s):
    net, c = s["net"], s["c"]
    if c["call"] == "predict":
        return net.predict(s["X"])
    if c["call"] == "forward":
        return net.forward_dev(c["rows"])
    net.train_step(c["rows"], s["T"], s["w"])
    return {"W": list(net.W), "b": list(net.b)}


# ---- the protocol ------------------------------------------------------------------------------
def prepare(case, seed):
    return {"cell": _prepare_cell, "batch": _prepare_batch, "mlp": _prepare_mlp}[case["kind"]](case, seed)


def run(state):
    return {"cell": _run_cell, "batch": _run_batch, "mlp": _run_mlp}[state["c"]["kind"]](state)


def work(case):
    """Bytes and operations of one pass.  A step reads and writes displacement and velocity state (48 B per
    node), reads the reference positions (12 B per node) and the corners (16 B per tetra); a law's own
    state and outputs come on top.  Operations per tetra: shape and gradient 75, strain and invariants 70,
    stress 40, forces 60, a flow update 150."""
    if case["kind"] == "mlp":
        macs = sum(a * b for a, b in zip(SIZES[:-1], SIZES[1:]))
        rows = case["rows"]
        flops = 2.0 * rows * macs
        if case["call"] == "train":
            return {"flops": 3 * flops, "bytes": macs * 28.0 + rows * 4.0 * (SIZES[0] + SIZES[-1])}
        return {"flops": flops, "bytes": macs * 2.0 + rows * (2.0 * SIZES[0] + 4.0 * SIZES[-1])}
    if case["kind"] == "batch":
        size = [_ball(d["m"], d["seed"] % 4) for d in _population(case, 0)]
        N, T = sum(len(p) for p, _ in size), sum(len(t) for _, t in size)
        per_tetra, ops = (16 + 48, 395) if case["viscous"] else (16, 245)
        return {"bytes": float(case["steps"]) * (60 * N + per_tetra * T), "flops": float(case["steps"]) * ops * T}
    P, tets = _ball(case["m"], 1)
    N, T, n = len(P), len(tets), float(case["steps"])
    state = {"vp_hard": 80, "prony": 72 + 144}.get(case["law"], 0)
    once = 8.0 * T if case["stress"] else 0.0
    ops = {"vp_hard": 395, "vp_yield": 265, "prony": 300}.get(case["law"], 245)
    return {"bytes": n * (60 * N + (16 + state) * T) + once, "flops": n * ops * T}


# ---- the same in float64 -----------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _mv(A, b):  # (T, 3, 3) x (T, 3)
    return (A * b[:, None, :]).sum(-1)


def _mm(A, B):
    return (A[:, :, :, None] * B[:, None, :, :]).sum(2)


def _tr(A):
    return A[:, 0, 0] + A[:, 1, 1] + A[:, 2, 2]


def _cof(A):  # row i = row i+1 x row i+2
    return torch.stack([torch.linalg.cross(A[:, (i + 1) % 3], A[:, (i + 2) % 3]) for i in range(3)], 1)


def _inv(A):
    C = _cof(A)
    return C.transpose(1, 2) / (A[:, 0] * C[:, 0]).sum(-1)[:, None, None]


class _Exact:
    """Float64 steps of a set of cells: ``par`` holds per-tetra tensors (law constants) and per-node tensors (contacts)."""

    def __init__(self, X, tets, law, par):
        self.X, self.tets, self.law, self.par = X, tets, law, par
        self.ids = tets.T.reshape(-1)
        self.I = torch.eye(3, dtype=torch.float64, device=X.device)[None]
        Dm = self.edges(X)
        self.Dinv = _inv(Dm)
        self.six_v0 = (Dm[:, :, 0] * torch.linalg.cross(Dm[:, :, 1], Dm[:, :, 2])).sum(-1)
        T = len(tets)
        if law in ("vp", "vp_hard"):
            self.Q = torch.zeros(T, 3, 3, dtype=torch.float64, device=X.device)
            self.eps = torch.zeros(T, dtype=torch.float64, device=X.device)
        if law == "prony":
            self.h = [torch.zeros(T, 3, 3, dtype=torch.float64, device=X.device) for _ in par["w"]]
            self.dev_old = torch.zeros(T, 3, 3, dtype=torch.float64, device=X.device)

    def edges(self, x):  # columns r1, r2, r3
        p = x[self.tets]
        return (p[:, 1:] - p[:, :1]).transpose(1, 2)

    def isotropic(self, B, J):  # Mooney-Rivlin Cauchy stress
        p = self.par
        I1 = _tr(B)
        s = (p["mu1"] * J ** (-5 / 3))[:, None, None] * (B - I1[:, None, None] / 3 * self.I)
        if p["mr"]:
            M = I1[:, None, None] * B - _mm(B, B)
            s = s + (p["mu2"] * J ** (-7 / 3))[:, None, None] * (M - _tr(M)[:, None, None] / 3 * self.I)
        return s + (p["kappa"] * (J - 1))[:, None, None] * self.I

    def force(self, x):
        p, I = self.par, self.I
        F = I + _mm(self.edges(x - self.X), self.Dinv)
        C = _cof(F)
        J = (F[:, 0] * C[:, 0]).sum(-1)
        sgn = None
        if self.law in ("vp", "vp_hard"):
            Fe = _mm(F, I + self.Q)
            B = _mm(Fe, Fe.transpose(1, 2))
            sig = self.isotropic(B, torch.sqrt((B[:, 0] * _cof(B)[:, 0]).sum(-1)))
            dv = sig - _tr(sig)[:, None, None] / 3 * I
            svm = torch.sqrt(1.5 * (dv * dv).sum((1, 2)))
            over = torch.clamp(svm - p["sy"], min=0.0)
            s0 = p["Y"] * (1 + self.eps / p["eps0"]) ** p["n"] if self.law == "vp_hard" else p["Y"]
            rate = p["rate"] * (over / s0) ** p["m"] if self.law == "vp_hard" else p["rate"] * over / s0
            self.eps = self.eps + rate
            g = torch.where(svm > 0, 1.5 * rate / torch.clamp(svm, min=1e-300), torch.zeros_like(svm))
            self.Q = _mm(_inv(F), _mm(_inv(I + g[:, None, None] * dv), Fe)) - I
            sgn = torch.sign(self.six_v0 * J)
        elif self.law == "nh2":
            B = _mm(F, F.transpose(1, 2))
            Jb = J.abs()
            a = Jb ** (-5 / 3) * (p["mu1"] + p["mu2"] * (_tr(B) * Jb ** (-2 / 3) - 3))
            sig = a[:, None, None] * (B - _tr(B)[:, None, None] / 3 * I) + (p["kappa"] * (Jb - 1))[:, None, None] * I
            sgn = torch.sign(self.six_v0 * J)
        elif self.law == "prony":
            e = 0.5 * (F + F.transpose(1, 2)) - I
            dv = e - _tr(e)[:, None, None] / 3 * I
            sig = 2 * p["mu"] * (1 - sum(p["w"])) * dv + p["kappa"] * _tr(e)[:, None, None] * I
            for j, (w, tau) in enumerate(zip(p["w"], p["tau"])):
                self.h[j] = math.exp(-1 / tau) * self.h[j] + 2 * p["mu"] * w * (dv - self.dev_old)
                sig = sig + self.h[j]
            self.dev_old = dv
            sgn = torch.sign(self.six_v0 * J)
        elif self.law == "svk":  # rows -V0 mu Dm^-1 F^T (kappa tr(B - I) I + (B - I))
            Bd = _mm(F, F.transpose(1, 2)) - I
            M = p["lam_ratio"] * _tr(Bd)[:, None, None] * I + Bd
            rows = _mm(self.Dinv, _mm(F.transpose(1, 2), M)) * (-self.six_v0 / 6 * p["mu"])[:, None, None]
        else:
            sig = self.isotropic(_mm(F, F.transpose(1, 2)), J)
            sgn = torch.ones_like(J)
        if sgn is not None:
            self.sig = sig
            # edge cofactors c_k = det(Dm) cof(F) d_k, d_k row k of Dm^-1; f_k = -(1/6) sigma c_k
            c = _mm(self.Dinv, C.transpose(1, 2)) * self.six_v0[:, None, None]
            rows = _mm(c, sig) * (-sgn / 6)[:, None, None]
        fk = torch.cat([-rows.sum(1, keepdim=True), rows], 1).transpose(0, 1).reshape(-1, 3)
        return torch.zeros_like(x).index_add_(0, self.ids, fk)

    def indenter(self, x, pos):
        """The indenter's force on every node."""
        f = torch.zeros_like(x)
        if self.par["indenter"] == "sphere":
            r = x.clone()
            r[:, 1] -= pos
            d = r.norm(dim=1)
            return r * (CONTACT * torch.clamp(self.par["tip"] - d, min=0.0) / torch.clamp(d, min=1e-300))[:, None]
        f[:, 1] = -CONTACT * torch.clamp(x[:, 1] - pos, min=0.0)
        return f

    def run(self, x, first, steps, pos, every=None):
        """``steps`` damped velocity-Verlet steps from rest; ``every(step, x, indenter force)`` before each move."""
        v, fo = torch.zeros_like(x), torch.zeros_like(x)
        a, b = 1 - 0.5 * XI, 1 + 0.5 * XI
        for i in range(steps):
            f = self.force(x)
            t = self.indenter(x, pos(first + i))
            if every:
                every(i, x, t)
            f += t
            f[:, 1] += CONTACT * torch.clamp(self.par["wall"] - x[:, 1], min=0.0)
            v = (v * a + 0.5 * (f + fo)) / b
            x = x + v * a + 0.5 * f
            fo = f
        return x, v, fo


def _exact_cell(c, seed):
    P, tets = _ball(c["m"], 1)
    if len(tets) * c["steps"] > 6e8:
        return None
    dev = _dev()
    x, X = _start_positions(c, seed)
    cfg = _cell_config(c)
    cell, R = cfg["CELL"], float(c["m"])
    nu, ratio = cell["PoissonRatio"], cell["MooneyRivlinRatio"]
    p0 = cell["YoungsModulusSI"] / E_SIM
    mu = E_SIM / (2 * (1 + nu))
    law = {"vp_yield": "vp", "nh": "mr"}.get(c["law"], c["law"])
    par = {"mu": mu, "mu1": ratio * mu, "mu2": (1 - ratio) * mu, "kappa": E_SIM / (3 * (1 - 2 * nu)), "mr": ratio != 1.0,
           "lam_ratio": nu / (1 - 2 * nu), "indenter": c["indenter"], "tip": 0.4 * R, "wall": -R}
    if c["law"] == "vp_yield":
        par |= {"rate": 1e-5, "Y": 300.0 / p0, "sy": 200.0 / p0}
    elif c["law"] == "vp_hard":
        par |= {"rate": 1e-5, "Y": 2.5e-8 ** 0.5, "sy": 0.0, "m": 2.0, "n": 0.3, "eps0": 0.05}
    elif c["law"] == "nh2":
        par |= {"mu1": mu, "mu2": 0.4 * mu}
    elif c["law"] == "prony":
        par |= {"w": cell["ViscoelasticWeights"], "tau": cell["ViscoelasticRelaxationTimes"]}
    Xd, xd = torch.from_numpy(X).to(dev), torch.from_numpy(x).to(dev)
    if c["law"] != "prony":  # the fused step starts from the FP32 displacement
        xd = Xd + (xd - Xd).float().double()
    start = R + (0.4 * R if c["indenter"] == "sphere" else 0.0)
    pos = lambda t: start - R / 80000 * min(t, 20000)  # noqa: E731
    e = _Exact(Xd, torch.from_numpy(tets).to(dev), law, par)
    hist = []
    first = START[c["indenter"]]
    xe, v, fo = e.run(xd, first, c["steps"], pos, lambda i, x, t: hist.append(-t[:, 1].sum()) if c["hist"] else None)
    soa = lambda a: a.T.reshape(-1)  # noqa: E731
    out = {"x": soa(xe - Xd if c["law"] != "prony" else xe)}
    if c["steps"] <= FEW:
        out["v"], out["f"] = soa(v), soa(fo)
    if c["hist"]:
        out["hist"] = torch.stack(hist)
    if c["record"]:
        now = first + c["steps"]
        L0 = cell["RadiusSI"] / R
        f = -e.indenter(xe, pos(now))[:, 1].sum().item()
        out["row"] = torch.tensor([(pos(0) - pos(now)) * L0, f * p0 * L0 ** 2], dtype=torch.float64)
    if c["stress"]:
        dv = e.sig - _tr(e.sig)[:, None, None] / 3 * e.I
        out["stress"], out["pressure"] = torch.sqrt(1.5 * (dv * dv).sum((1, 2))), _tr(e.sig) / 3
    if c["law"] in ("vp_yield", "vp_hard"):
        out["plastic"], out["strain"] = e.Q.reshape(-1, 9).T.reshape(-1), e.eps
    elif c["law"] == "prony":
        out["transient"] = torch.cat([h.reshape(-1, 9).T.reshape(-1) for h in e.h])
    return out


def _exact_batch(c, seed):
    dev = _dev()
    pop = _population(c, seed)
    X, tets, node, tetra, off = [], [], [], [], 0
    for i, d in enumerate(pop):
        P, T = _ball(d["m"], d["seed"] % 4)
        M = E_SIM * (1 - d["nu"]) / ((1 + d["nu"]) * (1 - 2 * d["nu"]))
        d["Rs"] = float(d["m"]) * min(1.0, 0.075 / M)  # lattice spacing of at most one length, stable for this material
        P = P * (d["R"] / d["m"])
        X.append((P * (d["Rs"] / abs(P[1, 0]))).astype(np.float32).astype(np.float64))
        tets.append(T + off)
        node += [np.full(len(P), i)]
        tetra += [np.full(len(T), i)]
        off += len(P)
    if sum(map(len, tets)) * c["steps"] > 1.5e9:
        return None
    per = lambda k, at: torch.tensor([float(k(d)) for d in pop], dtype=torch.float64, device=dev)[at]  # noqa: E731
    Xd = torch.from_numpy(np.concatenate(X)).to(dev)
    node, tetra = (torch.from_numpy(np.concatenate(a)).to(dev) for a in (node, tetra))
    mu1 = per(lambda d: E_SIM / (2 * (1 + d["nu"])), tetra)
    par = {"mu1": mu1, "mr": False, "kappa": per(lambda d: E_SIM / (3 * (1 - 2 * d["nu"])), tetra), "indenter": "sphere",
           "tip": per(lambda d: d["tip"] / d["R"] * d["Rs"], node), "wall": per(lambda d: -d["Rs"], node),
           "rate": per(lambda d: d["T0"], tetra), "Y": per(lambda d: 3 * d["eta"] / (d["E"] / E_SIM), tetra), "sy": 0.0}
    Rs = per(lambda d: d["Rs"], node)
    e = _Exact(Xd, torch.from_numpy(np.concatenate(tets)).to(dev), "vp" if c["viscous"] else "mr", par)
    curves = torch.zeros(len(pop), c["ncurve"], dtype=torch.float64, device=dev)
    scale = torch.tensor([E_SIM * d["Rs"] ** 2 for d in pop], dtype=torch.float64, device=dev)

    def sample(i, x, t):
        k = i * c["ncurve"] // c["steps"]
        if i == 0 or (i - 1) * c["ncurve"] // c["steps"] != k:
            curves[:, k] = torch.zeros_like(scale).index_add_(0, node, -t[:, 1]) / scale

    xe, _, _ = e.run(Xd.clone(), 0, c["steps"], lambda t: Rs + par["tip"] - 0.3 * Rs / c["steps"] * t, sample)
    return {"curves": curves, "x": [(xe - Xd).T.reshape(-1)]}


def _exact_mlp(c, seed):
    dev = _dev()
    g = torch.Generator().manual_seed(seed % 1000)
    X, T, w = _network_inputs(c, seed)
    W, b = [], []
    for l, (fin, fout) in enumerate(zip(SIZES[:-1], SIZES[1:])):  # torch.nn.Linear's initial weights
        bound = 1.0 / math.sqrt(fin)
        W.append(((torch.rand(fout, fin, generator=g, dtype=torch.float64) * 2 - 1).float() * bound).double().to(dev))
        b.append(((torch.rand(fout, generator=g, dtype=torch.float64) * 2 - 1) * bound).float().double().to(dev))
    par = [t.requires_grad_(c["call"] == "train") for t in W + b]
    h = torch.from_numpy(X).double().to(dev)
    for l in range(len(W)):
        h = h @ W[l].T + b[l]
        if l < len(W) - 1:
            h = torch.nn.functional.gelu(h)
    if c["call"] != "train":
        return h
    loss = (torch.from_numpy(w).double().to(dev)[:, None] * (h - torch.from_numpy(T).double().to(dev)) ** 2).mean()
    loss.backward()
    t = ADAM_STEP + 1
    out = {"W": [], "b": []}
    with torch.no_grad():
        for l in range(len(W)):
            for name, p, s in (("W", W[l], 10 * seed + l), ("b", b[l], 10 * seed + 5 + l)):
                pad = -p.shape[-1] % 32 if name == "W" else 0
                shape = (p.shape[0], p.shape[1] + pad) if name == "W" else tuple(p.shape)
                m, v = (a.double() for a in _moments(shape, s, dev))
                new, grad = torch.nn.functional.pad(p, (0, pad)), torch.nn.functional.pad(p.grad, (0, pad))
                if pad:
                    m[:, p.shape[1]:] = 0
                m, v = 0.9 * m + 0.1 * grad, 0.999 * v + 0.001 * grad ** 2
                out[name].append(new - 1e-3 / (1 - 0.9 ** t) * m / (v.sqrt() / math.sqrt(1 - 0.999 ** t) + 1e-8))
    return out


def exact(case, seed):
    """What ``run`` returns on a fresh state, in float64."""
    return {"cell": _exact_cell, "batch": _exact_batch, "mlp": _exact_mlp}[case["kind"]](case, seed)
