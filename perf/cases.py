"""The workloads whose speed is watched: what a user of the library runs.

A discharge case is created from a deck, stepped with ``Case.step`` and read
back every few steps, as a program does that follows a discharge (profiles,
collision counts, electron energies).  Several small cases step together
through ``Batch``; independent Poisson problems are solved through
``PoissonBatch``.
Everything goes through the package's public entry points.

A case here is a dict of plain values:

  kind "step"     one discharge, ``steps`` fused steps per pass, then a readout
  kind "batch"    ``cases`` argon discharges of different sizes in one Batch
  kind "poisson"  ``problems`` independent 5-point problems, right-hand sides
                  in, solutions out
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hybrid-final_amd"))

from picmcc import FP32_REFINED, FP64_PLAIN, Batch, Case, PoissonBatch, decks, poisson_cases  # noqa: E402

FIELDS = ("den", "phi", "Ex", "Ey")


def step_case(gas, precision, nx, ny, ppc, steps, name=None, solver=0, walls="ccp", read="fields", dx=2e-4,
              volts=150.0, torr=0.05, per_cycle=400, capacity=3.0):
    c = {"kind": "step", "gas": gas, "precision": precision, "nx": nx, "ny": ny, "ppc": ppc, "steps": steps,
         "solver": solver, "walls": walls, "read": read, "dx": dx, "volts": volts, "torr": torr,
         "per_cycle": per_cycle, "capacity": capacity}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest discharges of a parameter scan: a step is a chain of
        # short launches; the caller follows the electron energies
        step_case("ar", "f32", 32, 24, 20, 40, "ar 32x24 spectrum", dx=5e-4, torr=0.1, read="spectrum",
                  capacity=4.0),
        # the 64x64 argon benchmark deck, profiles and collision counts read
        # ten times an RF cycle
        step_case("ar", "f32", 64, 64, 50, 40, "ar 64x64", dx=5e-4, volts=100.0, torr=0.1, read="counts"),
        # an odd, tall grid of the size an ensemble serves, low pressure
        step_case("ar", "f32", 75, 181, 60, 12, "ar 75x181 tall", volts=220.0, torr=0.02),
        # the 256x256 argon benchmark deck (26 M particles)
        step_case("ar", "f32", 256, 256, 200, 8, "ar 256x256", volts=200.0, per_cycle=800, capacity=2.0),
        # double precision on the direct field solve: the reference run a
        # single-precision result is checked against
        step_case("ar", "f64", 128, 128, 100, 8, "ar f64 128x128", solver=2, volts=200.0, per_cycle=800),
        # the reference algorithm in double precision (Jacobi PCG), 64x64 deck
        step_case("ar", "f64", 64, 64, 50, 4, "ar f64 pcg 64x64", dx=5e-4, volts=100.0, torr=0.1, read="spectrum"),
        # a discharge confined by a dielectric side wall between thick
        # electrodes: the field operator is not separable
        step_case("ar", "f32", 128, 96, 60, 4, "ar dielectric 128x96", walls="dielectric", read="counts"),
        # oxygen chemistry, four species, the ions colliding
        step_case("o2", "f32", 192, 192, 50, 8, "o2 192x192", volts=100.0, per_cycle=800),
        # Ar/O2, five species: one of the small cases that are served by the
        # hundred, and a large one
        step_case("aro2", "f32", 72, 65, 24, 12, "aro2 72x65", torr=0.1, read="counts", capacity=4.0),
        step_case("aro2", "f32", 256, 128, 100, 8, "aro2 256x128", torr=0.03, per_cycle=800),
        # a dozen small discharges of a scan stepped together
        {"kind": "batch", "name": "batch of 12", "cases": 12, "lo": 24, "hi": 48, "ppc": 25, "steps": 30},
        # potentials of many charge distributions at once
        {"kind": "poisson", "name": "poisson 64", "problems": 64, "lo": 48, "hi": 224},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["ar", "ar", "ar", "f64", "pcg", "dielectric", "o2", "aro2", "batch", "poisson"])
    if kind == "batch":
        lo = rng.randint(16, 40)
        return {"kind": "batch", "cases": rng.randint(3, 16), "lo": lo, "hi": lo + rng.randint(4, 32),
                "ppc": rng.randint(10, 40), "steps": rng.randint(15, 30)}
    if kind == "poisson":
        lo = rng.randint(17, 100)
        return {"kind": "poisson", "problems": rng.randint(5, 80), "lo": lo, "hi": lo + rng.randint(1, 120)}
    # one side up to 288 cells, the other at most 160 (the host setup's
    # direct solves grow with the cube of the short side)
    side = {"pcg": 72, "dielectric": 112, "f64": 144}.get(kind, 288)
    nx, ny = int(_log(rng, 20, side)), int(_log(rng, 20, min(side, 160)))
    if rng.random() < 0.4 and nx <= 160:
        nx, ny = ny, nx
    if kind == "dielectric":
        nx, ny = max(nx, 24), max(ny, 24)
    most = {"pcg": 4e5, "dielectric": 1.5e6, "f64": 3e6, "o2": 5e6, "aro2": 8e6}.get(kind, 1.2e7)
    ppc = int(max(10, min(_log(rng, 12, 200), most / (2 * nx * ny))))
    per = {"ar": 2, "f64": 2, "pcg": 2, "dielectric": 2, "o2": 2.4, "aro2": 3.4}[kind] * ppc * nx * ny
    if kind in ("pcg", "dielectric"):
        steps = rng.randint(2, 4)
    else:
        steps = max(4, min(40, int(1.2e7 / per) + rng.randint(0, 4)))
    # gaps of at least a centimetre, where the plasma holds, and at most 15 kV/m
    dx = rng.choice([2e-4, 5e-4]) if ny >= 64 else 5e-4
    kw = {"dx": dx, "volts": float(min(rng.randint(50, 300), int(15e3 * ny * dx))), "torr": _log(rng, 0.01, 0.4),
          "per_cycle": rng.choice([400, 800]), "read": rng.choice(["fields", "counts", "spectrum"]), "capacity": 4.0}
    if kind == "f64":
        return step_case("ar", "f64", nx, ny, ppc, steps, solver=2, **kw)
    if kind == "pcg":
        return step_case("ar", "f64", nx, ny, ppc, steps, **kw)
    if kind == "dielectric":
        return step_case("ar", rng.choice(["f32", "f32", "f64"]), nx, ny, ppc, steps,
                         walls="dielectric", **kw)
    return step_case(kind, "f32", nx, ny, ppc, steps, **kw)


def _deck(c, seed):
    rng = random.Random(seed)
    kw = dict(ncx=c["nx"], ncy=c["ny"], dx=c["dx"], volts=c["volts"], pres_torr=c["torr"], ppc=c["ppc"],
              steps_per_cycle=c["per_cycle"], capacity_factor=c["capacity"], seed=rng.randrange(1, 1 << 30),
              philox_seed=rng.randrange(1, 1 << 40))
    if c["gas"] == "o2":
        d = decks.oxygen_deck(gas=1, ion_collisions=True, **kw)
    elif c["gas"] == "aro2":
        d = decks.oxygen_deck(gas=2, o2_ratio=0.2, **kw)
    else:
        d = decks.ccp_deck(**kw)
    geo = d["Geometry"]
    # the RF phase at which the run starts
    geo["Source"][0]["Phase(deg)"] = rng.uniform(0.0, 360.0)
    if c["walls"] == "dielectric":
        ny, nx = c["ny"], c["nx"]
        geo["ConductorSpec"][0].update({"Y0": ny - 2, "Y1": ny})
        geo["ConductorSpec"][1].update({"Y0": 0, "Y1": 1})
        geo["DielectricSpec"] = [{"M_ID": 3, "X0": 3 * nx // 4, "X1": nx, "Y0": 1, "Y1": ny - 2, "Epsilon": 4.0}]
    return d


def _batch_decks(c, seed):
    rng, shape = random.Random(seed), random.Random(c["cases"] * 1000 + c["lo"])
    out = []
    for _ in range(c["cases"]):
        nx, ny = shape.randint(c["lo"], c["hi"]), shape.randint(c["lo"], c["hi"])
        out.append(decks.ccp_deck(ncx=nx, ncy=ny, dx=5e-4, volts=shape.uniform(60, 250),
                                  pres_torr=math.exp(shape.uniform(math.log(0.03), math.log(0.3))),
                                  ppc=c["ppc"] + shape.randint(0, 10), steps_per_cycle=400, capacity_factor=4.0,
                                  seed=rng.randrange(1, 1 << 30), philox_seed=rng.randrange(1, 1 << 40)))
    return out


def _poisson(c, seed):
    """Sizes and walls of the problems (the plan) and right-hand sides of `seed`."""
    sizes, bcs = [], []
    shape = random.Random(c["problems"] * 1000 + c["lo"])
    for _ in range(c["problems"]):
        sizes.append(tuple(int(round(_log(shape, c["lo"], c["hi"]))) for _ in range(2)))
        bcs.append(poisson_cases.BC_PATTERNS[shape.randrange(len(poisson_cases.BC_PATTERNS))])
    rng = np.random.default_rng(seed)
    rhs = []
    for nx, ny in sizes:
        rho = rng.uniform(-1e-5, 1e-5, size=(nx, ny))
        for _ in range(int(rng.integers(1, 9))):
            w = rng.uniform(2, 20)
            gx = np.exp(-((np.arange(nx) - rng.uniform(0, nx)) ** 2) / (2 * w * w))
            gy = np.exp(-((np.arange(ny) - rng.uniform(0, ny)) ** 2) / (2 * w * w))
            rho += rng.normal(0.0, 1e-3) * gx[:, None] * gy[None, :]
        rhs.append((rho * 4e-8 / poisson_cases.EPS0).ravel())
    return sizes, bcs, np.concatenate(rhs)


def prepare(case, seed):
    if case["kind"] == "batch":
        cs = [Case(d, FP32_REFINED) for d in _batch_decks(case, seed)]
        return {"case": case, "cases": cs, "batch": Batch(cs)}
    if case["kind"] == "poisson":
        sizes, bcs, rhs = _poisson(case, seed)
        return {"case": case, "solver": PoissonBatch(sizes, bcs), "rhs": rhs}
    prec = FP64_PLAIN if case["precision"] == "f64" else FP32_REFINED
    return {"case": case, "sim": Case(_deck(case, seed), prec, field_solver=case["solver"])}


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        state["batch"].step(case["steps"])
        return [{f: c.array(f) for f in ("den", "phi", "mccr")} for c in state["cases"]]
    if case["kind"] == "poisson":
        solver = state["solver"]
        solver.set_rhs(state["rhs"])
        solver.solve(1e-10, 3)
        x, _, bad = solver.result()
        return {"x": x, "unsolved": bad}
    sim = state["sim"]
    sim.step(case["steps"])
    if case["read"] == "spectrum":
        sim.eedf_sample(60.0)
    out = {f: sim.array(f) for f in FIELDS}
    info = sim.info()
    out["np"] = np.array(info.np[:info.nsp], dtype=np.float64)
    if case["read"] != "fields":
        out["mccr"] = sim.array("mccr")
    if case["read"] == "spectrum":
        out["eedf"] = sim.array("eedf")
    return out


def _species(c):
    """Particles per cell of each species."""
    low = max(1, c["ppc"] // 5)
    return {"ar": [c["ppc"]] * 2, "o2": [c["ppc"], c["ppc"], low, low],
            "aro2": [c["ppc"]] * 3 + [low] * 2}[c["gas"]]


def _step_work(nx, ny, per_cell, steps, real):
    """Each step reads and writes every particle record once (five reals and
    an id), and the node fields (density, potential, field) once; the push
    takes about 50 operations, a collision test about 100, the direct field
    solve four matrix products."""
    n = sum(per_cell) * nx * ny
    nodes = (nx + 1) * (ny + 1)
    return (steps * (2.0 * n * (5 * real + 4) + nodes * real * (len(per_cell) + 4)),
            steps * (150.0 * n + 4.0 * nodes * (nx + ny)))


def work(case):
    if case["kind"] == "poisson":
        n, f = 0, 0
        for nx, ny in _poisson(case, 1)[0]:
            n += nx * ny
            f += 4 * nx * ny * (nx + ny)
        return {"bytes": 16.0 * n, "flops": float(f)}
    if case["kind"] == "batch":
        b, f = 0.0, 0.0
        for d in _batch_decks(case, 1):
            s = d["Geometry"]["SystemSpec"]
            w = _step_work(s["NumGridx"] - 1, s["NumGridy"] - 1, [case["ppc"] + 5] * 2, case["steps"], 4)
            b, f = b + w[0], f + w[1]
        return {"bytes": b, "flops": f}
    real = 8 if case["precision"] == "f64" else 4
    b, f = _step_work(case["nx"], case["ny"], _species(case), case["steps"], real)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Four times the spread seen when the first right-hand side of a pass was
    changed in its last bits, as another order of the deposit's sums or
    another solver at the deck's 1e-10 would, over five seeds of each listed
    case.  In single precision that now and then turns one particle's
    collision, which a node of some tens of particles shows (largest
    difference seen: 1.7e-3 in Ex, which is noise about 0, 4.6e-2 at a node);
    the direct solve in double precision stays within 1.3e-13, the PCG's
    stopping rule within 4e-9.  The Poisson problems lie within 4.5e-12 of
    exact()."""
    if case["kind"] == "poisson":
        return {"rel": 2e-11, "max": 2e-10}
    if case["kind"] == "step" and case["precision"] == "f64":
        if case["solver"] == 2 and case["walls"] == "ccp":
            return {"rel": 1e-12, "max": 1e-11, "differ": 1e-4}
        return {"rel": 2e-8, "max": 2e-7, "differ": 1e-4}
    return {"rel": 5e-3, "max": 0.15, "differ": 1e-3}


def exact(case, seed):
    """Poisson problems: the separable operator's inverse by eigenvectors, in
    64 bits.  A discharge step has no closed form."""
    if case["kind"] != "poisson":
        return None
    sizes, bcs, rhs = _poisson(case, seed)

    def basis(n, left, right):
        t = 2.0 * torch.eye(n, dtype=torch.float64)
        i = torch.arange(n - 1)
        t[i, i + 1] = -1.0
        t[i + 1, i] = -1.0
        w = torch.ones(n, dtype=torch.float64)   # a mirror row is twice its half cell
        if left == 0:
            t[0, 1], w[0] = -2.0, 0.5
        if right == 0:
            t[n - 1, n - 2], w[n - 1] = -2.0, 0.5
        h = torch.sqrt(w)
        lam, q = torch.linalg.eigh(h[:, None] * t / h[None, :])
        return lam, q / h[:, None], q.T * h[None, :]

    out, at = [], 0
    for (nx, ny), (l, r, b, t) in zip(sizes, bcs):
        lx, vx, vxi = basis(nx, l, r)
        ly, vy, vyi = basis(ny, b, t)
        f = torch.from_numpy(rhs[at:at + nx * ny].reshape(nx, ny))
        at += nx * ny
        out.append((vx @ ((vxi @ f @ vyi.T) / (lx[:, None] + ly[None, :])) @ vy.T).reshape(-1))
    return {"x": torch.cat(out), "unsolved": None}
