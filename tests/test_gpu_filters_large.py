"""The filter loops where a grid has more tiles than compute units (every tile
of the next launch then reduces more partial maxima than it preloads), more
than are reduced by every tile (k_filter_reduce), and on the narrowest grids
with an isothermal bottom, whose wall rows take thresholds above their fixed
step.  Against the loop with a host round trip per check (PT_FILTER_HOST=1):
the same arithmetic, so the pass counts and the fields are equal."""
import numpy as np
import pytest

from projectracer_amd import Simulation, cases

pytestmark = pytest.mark.gpu


def _run(case, monkeypatch, host):
    monkeypatch.setenv("PT_FILTER_HOST", "1" if host else "0")
    sim = Simulation(case.params)
    assert (sim.nx, sim.nz) == (case.nx, case.nz)
    sim.load_state(case)
    sim.tracers_to_corners()
    inf = sim.info()
    out = (inf["n_comp"], inf["n_temp"]), sim.field("TVIS").copy(), sim.field("CVIS").copy()
    sim.close()
    return out


@pytest.mark.parametrize("nx,nz,tpc,grids,dT,dC,fewest", [
    (2048, 512, 1, 6, 1.03, 1.05, (20, 1)),    # 512 tiles of each loop
    (1984, 1984, 1, 6, 1.03, 1.05, (20, 1)),   # 1278 (T) and 1534 (C) tiles
    (8, 8, 6, 2, 1.6, 1.05, (1, 1)),
    (24, 10, 6, 2, 1.45, 1.05, (1, 1)),
    (12, 24, 6, 2, 1.2, 1.05, (1, 1)),
])
def test_filters_equal_the_host_loop(nx, nz, tpc, grids, dT, dC, fewest, monkeypatch):
    print(f"[filters] {nx}x{nz}", flush=True)
    case = cases.thermochem(nx=nx, nz=nz, tpc=tpc, aspect=nx / nz, visT=30.0, visC=0.5, delta_visT=dT, delta_visC=dC,
                            grids=grids, mingrid=2)
    device, host = _run(case, monkeypatch, False), _run(case, monkeypatch, True)
    print(device[0], host[0], flush=True)
    assert device[0] == host[0] and host[0][0] >= fewest[0] and host[0][1] >= fewest[1]
    assert np.array_equal(device[1], host[1]) and np.array_equal(device[2], host[2])
