"""The RKC1 sweeps' results do not depend on their tiling: one cold solve with
at most 1, 2, 3 and 5 stages per launch (PT_SWEEP_STAGES; the tile and the rows
per thread change with it) against the tiling the library takes by itself, bit
for bit, on levels of one tile, of several, ragged ones and tiny ones, for both
operators and both precisions (rigid walls in FP64, where they converge)."""
import numpy as np
import pytest

from projectracer_amd import Simulation, _abi, cases

pytestmark = pytest.mark.gpu

GRIDS = [
    dict(nx=24, nz=24, grids=4, mingrid=3), dict(nx=66, nz=66), dict(nx=264, nz=24, aspect=11.0, grids=3),
    dict(nx=96, nz=48, aspect=2.0, Vbc=1), dict(nx=64, nz=32, aspect=2.0, Nmulti=2, nstageS=20),
    dict(nx=256, nz=128, aspect=2.0),
]


def _solve(case, monkeypatch, stages):
    monkeypatch.setenv("PT_SWEEP_STAGES", str(stages))
    sim = Simulation(case.params)
    sim.load_state(case)
    sim.multigrid()
    inf = sim.info()
    out = inf["q"], inf["residual"], sim.field("SF").copy()
    sim.close()
    return out


@pytest.mark.parametrize("law", ["iso", "law"])
@pytest.mark.parametrize("grid,precision", [(g, p) for g in GRIDS for p in ("fp64", "mixed")
                                            if p == "fp64" or not g.get("Vbc")],
                         ids=lambda v: v if isinstance(v, str) else f"{v['nx']}x{v['nz']}")
def test_sweeps_do_not_depend_on_the_tiling(grid, law, precision, monkeypatch):
    print(f"[tiling] {grid} {law} {precision}", flush=True)
    over = dict(grid, tpc=6, precision=_abi.PT_PREC_FP64 if precision == "fp64" else _abi.PT_PREC_MIXED)
    over.setdefault("aspect", 1.0)
    if precision == "mixed":
        over["tolerance"] = 1e-7
    if law == "iso":
        case = cases.isoviscous(nx=over.pop("nx"), nz=over.pop("nz"), tpc=over.pop("tpc"), **over)
    else:
        case = cases.thermochem(visT=10.0, visC=0.5, RaT=1e5, RaC=3e4, delta_visT=1.2, delta_visC=1.2, **over)
    q, res, psi = _solve(case, monkeypatch, 0)
    assert np.any(psi != 0.0)
    for stages in (1, 2, 3, 5):
        got = _solve(case, monkeypatch, stages)
        assert got[:2] == (q, res) and np.array_equal(got[2], psi), stages
