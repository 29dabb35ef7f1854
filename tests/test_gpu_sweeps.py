"""RKC1 sweeps with several stages per launch (k_sweep) where their tiling can
go wrong: levels of fewer than 7 cells (a point with ghost images beyond both
walls), levels one tile covers, partial tiles, grid powers that are not powers
of two, rigid walls, several sweeps per visit and the reference's other stage
counts.  One cold solve against the oracle: the cycle count is exact and psi
agrees to 1e-10, the tolerance every FP64 solve of this path is held to; the
mixed path reaches the stop test with psi within 1e-5 of the oracle's FP64
solve (both stop at a relative residual of 1e-8)."""
from fractions import Fraction

import numpy as np
import pytest

from projectracer_amd import PtError, Simulation, _abi, cases
from _support import OracleSim, rel_err

GRIDS = {
    "tiny levels": dict(nx=24, nz=24, grids=4, mingrid=3),
    "narrow": dict(nx=16, nz=64, aspect=0.25, grids=3, mingrid=2),
    "two levels": dict(nx=66, nz=66),
    "odd coarsest": dict(nx=176, nz=48, aspect=11 / 3),
    "wide": dict(nx=264, nz=24, aspect=11.0, grids=3),
    "rigid": dict(nx=96, nz=48, aspect=2.0, Vbc=1),
    "two sweeps": dict(nx=64, nz=32, aspect=2.0, Nmulti=2),
    "20 stages": dict(nx=64, nz=32, aspect=2.0, nstageS=20),
}


def _case(name, law, precision):
    over = dict(GRIDS[name], precision=precision, tpc=6)
    over.setdefault("aspect", 1.0)
    if law == "iso":
        return cases.isoviscous(nx=over.pop("nx"), nz=over.pop("nz"), tpc=over.pop("tpc"), **over)
    return cases.thermochem(visT=10.0, visC=0.5, RaT=1e5, RaC=3e4, delta_visT=1.2, delta_visC=1.2, **over)


def _solve(sim, case):
    """(cycles, psi) of one cold solve, or the error that stops it."""
    try:
        sim.load_state(case)
        sim.multigrid()
    except PtError as e:
        return e.code, None
    return sim.info()["q"], np.asarray(sim.field("SF"))


@pytest.mark.gpu
@pytest.mark.parametrize("law", ["iso", "law"])
@pytest.mark.parametrize("name", list(GRIDS))
def test_sweeps_fp64(name, law):
    print(f"[sweeps] {name} {law} FP64", flush=True)
    case = _case(name, law, _abi.PT_PREC_FP64)
    q, psi = _solve(Simulation(case.params), case)
    qo, ref = _solve(OracleSim(case.params), case)
    assert q == qo
    if ref is not None:
        assert rel_err(psi, ref) <= 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("law", ["iso", "law"])
@pytest.mark.parametrize("name", [n for n in GRIDS if n not in ("rigid", "narrow")])
def test_sweeps_mixed(name, law):
    print(f"[sweeps] {name} {law} mixed", flush=True)
    case = _case(name, law, _abi.PT_PREC_MIXED)
    sim = Simulation(case.params)
    _, psi = _solve(sim, case)
    case.params.precision = _abi.PT_PREC_FP64
    _, ref = _solve(OracleSim(case.params), case)
    assert psi is not None and ref is not None
    inf = sim.info()
    assert inf["residual"] / inf["res_ref"] <= case.params.tolerance
    assert rel_err(psi, ref) <= 1e-5


def _fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def test_quotient_by_reciprocal_is_correctly_rounded():
    """The two-step quotient the FP64 stencils use for grid powers that are
    not powers of two equals IEEE division, here in exact arithmetic."""
    rng = np.random.default_rng(7)
    for d in [float(x) for x in (1 / 48) ** np.arange(1, 5)] + rng.uniform(1e-10, 1.0, 40).tolist():
        rd = 1.0 / d
        near = [float(np.nextafter(k * d, s)) for k in (1.0, 3.0, 7.0) for s in (-np.inf, np.inf)]
        for s in near + (rng.standard_normal(60) * 10.0 ** rng.integers(-6, 12, 60)).tolist():
            q = s * rd
            for _ in range(2):
                q = _fma(_fma(-q, d, s), rd, q)
            assert q == s / d
