"""The calls of this framework whose time matters, at the sizes they are used at.

`listed()` gives the fixed cases and `draw()` others of the same ranges; `prepare()` makes
what a user's program holds before the call, `run()` is one pass through the public entry
points, `exact()` the same outputs in 64 bits from the mathematics where they have a closed
form, and `work()` the bytes and operations of one pass that no implementation can avoid
(inputs read once, outputs written once).

A program of this framework creates a context per model case, loads a temperature field and
its tracers, and then steps it: one stream-function solve with velocities, then four RK4
tracer stages with a projection each and three more solves (`time_step`), and the diagnostics
row of the step (`stats`).  The kinds:

  step      one time step of a running simulation and its diagnostics row
  solve     one multigrid solve from psi = 0 (the first solve of a run, or after a restart)
  direct    one velocity update with the direct banded solver, its matrix factored before
  build     assembling and factoring the direct solver's matrix (once per grid)
  project   one projection of the tracers to the nodes with the filters that follow it
  ensemble  one step of every case of an ensemble on one GPU
"""
import math

import numpy as np
import torch

from projectracer_amd import Simulation
from projectracer_amd._abi import PT_PREC_FP64, PT_PREC_MIXED, default_params
from projectracer_amd.cases import Case
from projectracer_amd.ensemble import Ensemble

PREC = {"f64": PT_PREC_FP64, "mixed": PT_PREC_MIXED}


def _step(name, nx, nz, tpc, law, prec, courant, tol=1e-8, discrete=False):
    return {"name": name, "kind": "step", "nx": nx, "nz": nz, "tpc": tpc, "law": law, "prec": prec,
            "courant": courant, "tol": tol, "discrete": discrete}


def _solve(name, nx, nz, law, prec, tol):
    return {"name": name, "kind": "solve", "nx": nx, "nz": nz, "tpc": 8, "law": law, "prec": prec, "tol": tol}


def _project(name, nx, nz, tpc, courant, tol):
    return {"name": name, "kind": "project", "nx": nx, "nz": nz, "tpc": tpc, "law": "law", "prec": "mixed",
            "courant": courant, "tol": tol}


def listed():
    return [
        # the smallest configuration: 64x64, constant viscosity, FP64, 84,500 tracers
        _step("step_iso_64x64_f64", 64, 64, 20, "iso", "f64", 0.5),
        # discrete tracer types with the tracer redistribution on (equalize=1), FP64
        _step("step_equalize_256x128_f64", 256, 128, 20, "iso", "f64", 0.5, discrete=True),
        # the thermochemical configuration's grid and 2 M tracers, eta(T, C), mixed path
        _step("step_law_384x128_mixed", 384, 128, 40, "law", "mixed", 0.02),
        # the benchmark's grid and 13.2 M tracers, constant viscosity, mixed path
        _step("step_iso_1024x256_mixed", 1024, 256, 50, "iso", "mixed", 0.5, 1e-7),
        # the benchmark's law on its grid and 13.2 M tracers, mixed path, at the small Courant
        # factor of a resolved flow (the filters' pass counts then stay alike from step to step)
        _step("step_law_1024x256_mixed", 1024, 256, 50, "law", "mixed", 0.05, 1e-7),
        # a projection of that workload at its own Courant factor, three steps into the run: 13.2 M
        # tracers that moved by several cells, and a composition field that needs a thousand passes
        # of its filter; every step makes four of them
        _project("project_law_1024x256", 1024, 256, 50, 0.25, 1e-7),
        # the first solve of the benchmark's law, mixed path
        _solve("solve_law_1024x256_mixed", 1024, 256, "law", "mixed", 1e-7),
        # the first solve on the full grid in plain FP64 (the reference's W-cycle)
        _solve("solve_iso_1024x256_f64", 1024, 256, "iso", "f64", 1e-7),
        # a first solve of the law in plain FP64 on a quarter-size grid
        _solve("solve_law_256x64_f64", 256, 64, "law", "f64", 1e-8),
        # the reference's shipped default: 100x100, direct solver; one velocity update
        {"name": "direct_100x100", "kind": "direct", "nx": 100, "nz": 100, "tpc": 8, "db": 2},
        # and the factorization that a run begins with
        {"name": "build_100x100", "kind": "build", "nx": 100, "nz": 100, "tpc": 8, "db": 2},
        # eight independent cases of different grids stepped together, mixed path
        {"name": "ensemble_8_mixed", "kind": "ensemble", "n": 8, "scale": 64, "tpc": 30},
    ]


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def _grid(rng, lo=32, hi=256):
    """nz a multiple of 16 (odd multiples among them) and nx = 1..4 times it: grids that
    optimize_grid leaves as they are."""
    nz = 16 * max(lo // 16, min(hi // 16, round(_log(rng, lo, hi) / 16)))
    return nz * rng.randint(1, 4), nz


def draw(rng):
    kind = rng.choice(["step", "step", "step", "solve", "solve", "project", "direct", "build", "ensemble"])
    if kind == "step":
        law, prec = rng.choice(["iso", "law"]), rng.choice(["f64", "mixed"])
        nx, nz = _grid(rng, 32, 128 if prec == "f64" else 256)
        discrete = law == "iso" and rng.random() < 0.25
        c = _step("", nx, nz, int(_log(rng, 8, 51)), law, prec, 0.02 if law == "law" else rng.choice([0.1, 0.5]),
                  1e-7 if nz > 128 else 1e-8, discrete)
    elif kind == "solve":
        law, prec = rng.choice(["iso", "law"]), rng.choice(["f64", "mixed"])
        nx, nz = _grid(rng, 32, 128 if prec == "f64" and law == "law" else 256)
        c = dict(_solve("", nx, nz, law, prec, 1e-7 if nz > 128 else 1e-8), tpc=int(_log(rng, 9, 31)))
    elif kind in ("direct", "build"):
        c = {"kind": kind, "nx": rng.randint(24, 100), "nz": rng.randint(24, 100), "tpc": rng.randint(6, 20),
             "db": rng.choice([1, 2])}
    elif kind == "project":
        nx, nz = _grid(rng, 48, 256)
        c = _project("", nx, nz, int(_log(rng, 8, 51)), 0.1, 1e-7)
    else:
        c = {"kind": kind, "n": rng.randint(2, 8), "scale": 16 * rng.randint(2, 4), "tpc": rng.randint(10, 30)}
    c.pop("name", None)
    return c


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
RAYLEIGH = {"iso": (1e5, 0.0), "discrete": (1e5, 5e4), "law": (1e6, 3e5)}


def _params(case):
    """The namelist values of one case."""
    nx, nz = case["nx"], case["nz"]
    kind = case["kind"]
    over = {"aspect": nx / nz, "nx": nx, "nz": nz, "tpc": case["tpc"], "grids": 6,
            "courant": case.get("courant", 0.5), "tolerance": case.get("tol", 1e-8),
            "precision": PREC[case.get("prec", "f64")]}
    over["RaT"], over["RaC"] = RAYLEIGH["discrete" if case.get("discrete") else case.get("law", "iso")]
    if nz >= 256:   # the full-size workload
        over["RaT"], over["RaC"] = 1e7, 3e6
    if case.get("law") == "law":
        over.update(ivis=2, visT=30.0, visC=0.5, delta_visT=1.2, delta_visC=1.2)
    if case.get("discrete"):
        over.update(iC_continuous=0, equalize=1, original=1, buffer=10)
    if kind in ("direct", "build"):
        over.update(iterate=0, Database=case["db"])
    return default_params(**over)


def _modes(seed):
    return 0.01 * np.random.default_rng(seed).standard_normal(8)


def _temp(a, x, z, aspect):
    acc = torch.zeros_like(x)
    for k in range(1, 9):
        acc += a[k - 1] * torch.cos(k * math.pi * x / aspect)
    return (1.0 - z) + acc * torch.sin(math.pi * z)


def _tensors(nx, nz, tpc, seed, layered):
    """Node temperatures and tracers (r, s, T, C) in ID order, on the GPU: tpc tracers per node
    placed uniformly in its dual cell, clamped to the walls; a two-layer composition at
    z = 0.3 or none."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    aspect = nx / nz
    dr, ds = aspect / nx, 1.0 / nz
    g = torch.Generator(device=dev).manual_seed(int(seed))
    a = _modes(seed)
    f8 = {"dtype": torch.float64, "device": dev}
    z, x = torch.meshgrid(ds * torch.arange(nz + 1, **f8), dr * torch.arange(nx + 1, **f8), indexing="ij")
    T = _temp(a, x, z, aspect)
    T[0, :] = 1.0
    T[nz, :] = 0.0
    shape = (nx + 1, nz + 1, tpc)
    i = torch.arange(nx + 1, **f8).reshape(-1, 1, 1)
    k = torch.arange(nz + 1, **f8).reshape(1, -1, 1)
    r = ((i + (torch.rand(shape, generator=g, **f8) - 0.5)) * dr).clamp_(0.0, aspect).reshape(-1)
    s = ((k + (torch.rand(shape, generator=g, **f8) - 0.5)) * ds).clamp_(0.0, 1.0).reshape(-1)
    Tt = _temp(a, r, s, aspect)
    if layered:
        Ct = (s < 0.3 + 0.01 * torch.cos(2.0 * math.pi * r / aspect)).to(torch.float64)
    else:
        Ct = torch.zeros_like(s)
    return T, r, s, Tt, Ct


def _layered(params):
    return params.RaC != 0.0


def _inputs(params, seed):
    T, r, s, Tt, Ct = (t.cpu().numpy() for t in _tensors(params.nx, params.nz, params.tpc, seed, _layered(params)))
    return Case("generated", params, T, 1.0, 0.0, r, s, Tt, Ct)


def _ensemble_params(case):
    """Grids of the ensemble configuration (128x64 to 384x128 at scale 64) with eta = exp(-gamma T)."""
    h = case["scale"]
    grids = [(2 * h, h), (3 * h, h), (4 * h, 2 * h), (6 * h, 2 * h)]
    out = []
    for j in range(case["n"]):
        nx, nz = grids[j % 4]
        RaT = 1e5 * 10.0 ** (j / 8)
        out.append(default_params(aspect=nx / nz, nx=nx, nz=nz, tpc=case["tpc"], grids=6, RaT=RaT, RaC=0.3 * RaT,
                                  ivis=1, visT=math.exp(0.4 * j), visP=1.0, delta_visT=2.0, delta_visC=2.0,
                                  courant=0.01, precision=PT_PREC_MIXED))
    return out


# --------------------------------------------------------------------------
# the measured calls
# --------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        ps = _ensemble_params(case)
        ens = Ensemble(ps)
        for j, (sim, p) in enumerate(zip(ens.cases, ps)):
            sim.load_state(_inputs(p, seed + 1000 * j))
        ens.run_steps(1, workers=case["n"])
        return {"kind": kind, "ens": ens, "workers": case["n"]}
    p = _params(case)
    sim = Simulation(p)
    if (sim.nx, sim.nz) != (p.nx, p.nz):
        raise ValueError("optimize_grid changed the grid to %dx%d" % (sim.nx, sim.nz))
    sim.load_state(_inputs(p, seed))
    state = {"kind": kind, "sim": sim}
    if kind == "step":
        sim.time_step()   # the simulation runs: its first, cold solve is behind it
    elif kind == "project":
        sim.run_steps(3)
    elif kind == "solve":
        state["psi0"] = np.zeros((p.nz + 7, p.nx + 7))
    elif kind == "direct":
        sim.build_sf_matrix()
    return state


def run(state):
    kind = state["kind"]
    if kind == "ensemble":
        status = state["ens"].run_steps(1, workers=state["workers"])
        out = {"status": status}
        for j, sim in enumerate(state["ens"].cases):
            out["T%d" % j], out["SF%d" % j] = sim.field("T"), sim.field("SF")
            out["nempty%d" % j] = sim.nempty()
        return out
    sim = state["sim"]
    if kind == "step":
        sim.time_step()
        row = sim.stats()
        return {"SF": sim.field("SF"), "T": sim.field("T"), "C": sim.field("CNEW"), "U": sim.field("U"),
                "W": sim.field("W"), "nempty": sim.nempty(),
                "stats": {k: row[k] for k in ("time", "Tavg", "vrms", "Nu", "Nu_bot", "Cavg")}}
    if kind == "project":
        sim.tracers_to_corners()
        return {"T": sim.field("T"), "C": sim.field("CNEW"), "Tvis": sim.field("TVIS"), "Cvis": sim.field("CVIS"),
                "nempty": sim.nempty()}
    if kind == "solve":
        sim.set_field("SF", state["psi0"])
        sim.multigrid()
        return {"SF": sim.field("SF")}
    if kind == "build":
        # psi of the first solve with the new factors: what a program goes on with
        sim.build_sf_matrix()
        sim.solve_sf_equation()
        return {"SF": sim.field("SF")}
    sim.update_velocities()
    return {"SF": sim.field("SF"), "U": sim.field("U"), "W": sim.field("W")}


# --------------------------------------------------------------------------
# 64-bit values
# --------------------------------------------------------------------------
def _exact_psi(p, seed):
    """psi of the discrete constant-viscosity problem by sine transforms: with free-slip walls
    psi is odd about every wall, so the fourth-order stencils are diagonal on sine modes."""
    nx, nz = p.nx, p.nz
    aspect = nx / nz
    dr, ds = aspect / nx, 1.0 / nz
    T0, r, s, Tt, Ct = _tensors(nx, nz, p.tpc, seed, _layered(p))
    dev = T0.device
    # tracer averages with bilinear weights at the nodes
    fi, fk = r / dr, s / ds
    i0, k0 = fi.floor().clamp(max=nx - 1), fk.floor().clamp(max=nz - 1)
    sums = torch.zeros(3, (nx + 1) * (nz + 1), dtype=torch.float64, device=dev)
    for di in (0, 1):
        for dk in (0, 1):
            w = (1.0 - (fi - (i0 + di)).abs()) * (1.0 - (fk - (k0 + dk)).abs())
            at = ((k0 + dk) * (nx + 1) + (i0 + di)).long()
            for j, v in enumerate((w * Tt, w * Ct, w)):
                sums[j].index_add_(0, at, v)
    T, C, w = (x.reshape(nz + 1, nx + 1) for x in sums)
    T = torch.where(w > 0, T / w, T0)
    C = torch.where(w > 0, C / w, torch.zeros_like(C))

    def ddx(f):   # fourth-order d/dx at the interior nodes, f even about the side walls
        e = torch.cat([f[:, [2, 1]], f, f[:, [nx - 1, nx - 2]]], dim=1)
        d = (e[:, :-4] - 8.0 * e[:, 1:-3] + 8.0 * e[:, 3:-1] - e[:, 4:]) / 12.0
        return d[1:nz, 1:nx] / dr

    rhs = p.RaT * ddx(T) - p.RaC * ddx(C)

    def basis(n, h):
        j = torch.arange(1, n, dtype=torch.float64, device=dev)
        th = math.pi * j / n
        d2 = (-5.0 / 2 + 8.0 / 3 * torch.cos(th) - 1.0 / 6 * torch.cos(2 * th)) / h ** 2
        d4 = (28.0 / 3 - 13.0 * torch.cos(th) + 4.0 * torch.cos(2 * th) - 1.0 / 3 * torch.cos(3 * th)) / h ** 4
        return torch.sin(math.pi / n * (torch.outer(j, j) % (2 * n))), d2, d4

    Sx, x2, x4 = basis(nx, dr)
    Sz, z2, z4 = basis(nz, ds)
    sym = x4[None, :] + z4[:, None] + 2.0 * z2[:, None] * x2[None, :]
    psi = Sz @ ((Sz @ rhs @ Sx) / sym) @ Sx * (4.0 / (nx * nz))
    out = np.zeros((nz + 7, nx + 7))
    inner = psi.cpu().numpy()
    for k in range(-3, nz + 4):
        kk, zs = (-k, -1.0) if k < 0 else (2 * nz - k, -1.0) if k > nz else (k, 1.0)
        if 1 <= kk <= nz - 1:
            out[k + 3, 4:nx + 3] = zs * inner[kk - 1]
    for q in range(1, 4):
        out[:, 3 - q] = -out[:, 3 + q]
        out[:, nx + 3 + q] = -out[:, nx + 3 - q]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("direct", "build") or (kind == "solve" and case["law"] == "iso"):
        out = {"SF": _exact_psi(_params(case), seed)}
        if kind == "direct":
            out["U"] = out["W"] = None
        return out
    return None


# --------------------------------------------------------------------------
# what one pass cannot do without
# --------------------------------------------------------------------------
def _step_work(nx, nz, ntr):
    nodes = (nx + 1) * (nz + 1)
    # tracers r, s, T read and written, C read; psi and T, C fields read and written, u, w written;
    # four RK4 stages interpolate three fields with a bicubic (about 40 operations each) and
    # project two values with bilinear weights (about 30); four operator applications
    return {"bytes": 56.0 * ntr + 64.0 * nodes, "flops": 4.0 * (150.0 * ntr + 80.0 * nodes)}


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        parts = [_step_work(p.nx, p.nz, (p.nx + 1) * (p.nz + 1) * p.tpc) for p in _ensemble_params(case)]
        return {k: sum(w[k] for w in parts) for k in ("bytes", "flops")}
    nx, nz = case["nx"], case["nz"]
    nodes = (nx + 1) * (nz + 1)
    if kind == "step":
        return _step_work(nx, nz, nodes * case["tpc"])
    if kind == "project":
        # tracers r, s, T, C read, T, C and their filtered copies written, nempty written; binning,
        # four bilinear weights and three weighted sums per tracer, one filter pass per field
        return {"bytes": 32.0 * nodes * case["tpc"] + 36.0 * nodes, "flops": nodes * (30.0 * case["tpc"] + 60.0)}
    if kind == "solve":
        # T, C and psi read, psi written; one operator application (the stop test)
        return {"bytes": 32.0 * nodes, "flops": 80.0 * nodes}
    kl = 3 * ((nx if case["db"] == 1 else nz) + 1)
    if kind == "direct":
        # the factors read once, T, C read, psi, u, w written; one multiply-add per factor entry
        return {"bytes": 8.0 * nodes * (3 * kl + 1) + 40.0 * nodes, "flops": 2.0 * nodes * 3 * kl}
    # the factors written once; a rank-1 update of kl x 2 kl per column
    return {"bytes": 8.0 * nodes * (3 * kl + 1), "flops": 4.0 * nodes * kl * kl}
