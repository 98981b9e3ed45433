"""The 2D gathers on row pieces, whose workgroups take particles and
candidate ranges from one table, against the direct gathers, bit for bit (same
neighbours, same order, same arithmetic).

Lattices with h = dx put every axis-aligned second neighbour at r = 2h,
jittered by 1e-6 dx, so that thousands of pairs straddle the cut-off that the
density pass pre-tests in 16-bit fixed point.  The row lengths end one short
of, at and one past a piece and leave fewer pieces than the workgroups are
dealt over; the dense ones hold more than 32 candidates in a row, and in
FP64 and FP32 more than a tile."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases

pytestmark = pytest.mark.gpu

# columns, rows, h / dx
LATTICES = {"one piece": (7, 3, 1.0), "short of a piece": (63, 9, 1.0),
            "pieces": (64, 18, 1.0), "past a piece": (65, 33, 1.0), "wide": (700, 6, 1.0),
            "masks overflow": (90, 40, 3.1), "tiles overflow": (80, 60, 5.3)}


@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
@pytest.mark.parametrize("name", list(LATTICES))
def test_piece_table_equals_direct(name, prec):
    nx, ny, h = LATTICES[name]
    c = cases.box_lattice(nx=nx, ny=ny, dx=0.01, jitter=1e-6, h_fac=h, precision=prec, vel=0.1)
    print(f"[gpu] piece table {name} n={c['n']} prec={prec}", flush=True)
    out = []
    for tiled in (True, False):
        sim = armando_amd.Simulation(c)
        sim.set_gather_path(tiled)
        sim.link_list()
        sim.density(0)
        sim.eos()
        sim.internal_force(c["flags"])
        r = dict(sim.rates())
        sim.time_integration(1, 2)
        out.append({**sim.state(), **{"r" + k: v for k, v in r.items()}})
        sim.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
