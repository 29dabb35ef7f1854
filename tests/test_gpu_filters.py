"""The filter loops with several passes per launch against the loop with a host
round trip per check (PT_FILTER_HOST=1, the reference's order,
PS/smoother.f90:582-672) where their tiles can go wrong: grids narrower than
the ghost columns' reach, one tile, partial tiles, grid powers that are not
powers of two, an insulating bottom with heating, pass counts on both sides of
a launch, and a field with an infinity.  The arithmetic per node and the
check are the same, so the pass counts and the filtered fields are equal."""
import numpy as np
import pytest

from projectracer_amd import PtError, Simulation, cases

pytestmark = pytest.mark.gpu

GRIDS = [(8, 8), (12, 24), (24, 10), (32, 64), (64, 32), (176, 48), (384, 128)]


def _run(case, monkeypatch, host):
    monkeypatch.setenv("PT_FILTER_HOST", "1" if host else "0")
    sim = Simulation(case.params)
    assert (sim.nx, sim.nz) == (case.nx, case.nz)
    try:
        sim.load_state(case)
        sim.tracers_to_corners()   # its first launch is sized by the first projection's counts
    except PtError as e:
        return e.code
    inf = sim.info()
    return inf["n_comp"], inf["n_temp"], sim.field("TVIS"), sim.field("CVIS")


@pytest.mark.parametrize("insulating", [0, 1])
@pytest.mark.parametrize("nx,nz", GRIDS)
def test_filters_equal_the_host_loop(nx, nz, insulating, monkeypatch):
    print(f"[filters] {nx}x{nz} insulating {insulating}", flush=True)
    for dT, dC in ((1.2, 1.2), (1.1, 1.05)):
        case = cases.thermochem(nx=nx, nz=nz, tpc=6, aspect=nx / nz, visT=30.0, visC=0.5, delta_visT=dT,
                                delta_visC=dC, Tbot=insulating, grids=2 if nz < 16 else 4, mingrid=2,
                                H=0.5 * insulating, Htype=2.0)
        if insulating == 0 and nz < 64 and dT < 1.2:
            continue   # the wall rows' fixed steps exceed this threshold: no loop ends
        if insulating == 0 and nz <= 24 and (nx, nz) != (12, 24):
            continue
        device, host = _run(case, monkeypatch, False), _run(case, monkeypatch, True)
        print(device[:2], host[:2])
        assert device[:2] == host[:2]
        assert np.array_equal(device[2], host[2]) and np.array_equal(device[3], host[3])


def test_filters_with_an_infinite_value(monkeypatch):
    case = cases.thermochem(nx=64, nz=32, tpc=6, aspect=2.0, visT=30.0, visC=0.5, delta_visT=1.2, delta_visC=1.2,
                            grids=4, mingrid=2)
    case.Ctr[1000] = np.inf
    device, host = _run(case, monkeypatch, False), _run(case, monkeypatch, True)
    assert device[:2] == host[:2]
    for d, h in zip(device[2:], host[2:]):
        assert np.array_equal(d, h, equal_nan=True)
