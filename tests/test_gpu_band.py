"""The band factorization and the band solves at the sizes where their code
changes: the numbers of rows a lane holds, matrices smaller than a panel of
columns or a block of rows, last panels and blocks that are partly filled, the
widest band (kl = 1023), both orderings of the nodes and rigid boundaries.
Same buoyancy fields on both sides; the operations are the oracle's, in its
order, so psi, u and w are compared bit for bit."""
import numpy as np
import pytest

from projectracer_amd import Simulation, cases, _abi
from _support import OracleSim, interior

pytestmark = pytest.mark.gpu

SIZES = [
    # nx, nz, Database, Vbc
    (8, 8, 1, 0), (8, 8, 2, 1), (9, 13, 1, 0), (9, 24, 2, 0), (24, 17, 1, 1), (40, 40, 2, 0),
    (36, 9, 1, 0), (37, 9, 1, 0),     # kl + 16 = 127, 130: 2 and 3 rows per lane
    (58, 8, 1, 0), (79, 8, 1, 0),     # 193, 256: 4
    (80, 8, 1, 0), (101, 8, 1, 0),    # 259: 5; 322: 6
    (122, 8, 1, 0), (123, 8, 1, 0),   # 385, 388: 8
    (165, 8, 1, 0), (207, 8, 1, 0),   # 514, 640: 10
    (208, 8, 1, 0),                   # 643: 13
    (272, 8, 1, 0), (10, 339, 2, 0),  # 835: 17; 1036
    (340, 8, 1, 0),                   # 1039: the widest band
]


@pytest.mark.parametrize("nx,nz,db,vbc", SIZES)
def test_band_solver_matches_the_oracle_bit_for_bit(nx, nz, db, vbc):
    print(f"[band] {nx}x{nz} Database {db} Vbc {vbc}: GPU vs oracle", flush=True)
    case = cases.isoviscous(nx=nx, nz=nz, tpc=1, aspect=nx / nz, iterate=0, Database=db, Vbc=vbc)
    gpu, ora = Simulation(case.params), OracleSim(case.params)
    gpu.load_state(case)
    ora.load_state(case)
    for n in ("TBUOY", "CBUOY"):
        gpu.set_field(n, ora.field(n))
    gpu.update_velocities()
    ora.update_velocities()
    for n in ("SF", "U", "W"):
        h = _abi.FIELD_HALO[_abi.FIELD[n]]
        a, b = interior(gpu.field(n), h, nx, nz), interior(ora.field(n), h, nx, nz)
        assert np.any(b != 0.0) and np.array_equal(a, b), n
