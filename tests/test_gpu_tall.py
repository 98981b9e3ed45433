"""2D grids of many cell rows (a standing pipe, a tall column): the table of row
pieces is made by workgroups of 256 rows' sums and, above 4096 rows, wavefronts of
several rows.  The tiled gathers on it equal the direct ones bit for bit, at row
counts around those limits, with few particles and with rows of several pieces;
and the table costs no more than the grid's other passes: the reorder pass of few
particles in 60,000 rows takes at most ten times that of the same particles in
48 rows of as many cells in all (26 us and 8 us as measured; 2,283 us when every
workgroup counted every row)."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases

pytestmark = pytest.mark.gpu


def column(nx, ny, prec, grid_ny, grid_nx=None, lift=0, gap=False):
    """A lattice block in a grid of grid_ny rows, `lift` cells above its own place; with
    gap, the particles of a band of columns taken out of every other dozen rows."""
    c = cases.box_lattice(nx=nx, ny=ny, dx=0.01, jitter=0.02, precision=prec, vel=0.1)
    if gap:
        keep = (np.abs(c["x"] - 0.005 * nx) > 0.004 * nx) | (c["y"] * 100 % 24 < 12)
        for k in ("x", "y", "vx", "vy", "rho", "u"):
            c[k] = c[k][keep]
        c["n"] = c["np"] = int(keep.sum())
    c["y"] = c["y"] + lift * c["cell"]
    c["ny"] = grid_ny
    if grid_nx:
        c["nx"] = grid_nx
    return c


# lattice columns and rows, grid rows, cells the block is lifted by, gap
GRIDS = {"one chunk": (30, 600, 256, 0, False), "past a chunk": (30, 600, 257, 0, False),
         "chunks": (30, 2500, 1100, 60, False), "one row a wavefront": (20, 300, 4096, 3900, False),
         "several rows": (20, 300, 4097, 3900, False), "partial share": (25, 9000, 9001, 5000, False),
         "gaps": (400, 500, 5000, 4700, True), "most rows": (24, 100, 65535, 65480, False),
         "tall": (40, 4000, 60000, 123, False)}


@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
@pytest.mark.parametrize("name", list(GRIDS))
def test_tall_grid_equals_direct(name, prec):
    nx, ny, gy, lift, gap = GRIDS[name]
    c = column(nx, ny, prec, gy, lift=lift, gap=gap)
    print(f"[gpu] tall grid {name} n={c['n']} {c['nx']}x{gy} prec={prec}", flush=True)
    out = []
    for tiled in (True, False):
        sim = armando_amd.Simulation(c)
        sim.set_gather_path(tiled)
        sim.link_list()
        sim.single_step()
        r = dict(sim.rates())
        sim.time_integration(1, 3)
        out.append({**sim.state(), **{"r" + k: v for k, v in r.items()}})
        sim.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k


def test_table_cost_of_many_rows():
    us = {}
    for name, gx, gy in (("tall", 20, 60000), ("wide", 25000, 48)):
        c = column(24, 100, cases.FP32, gy, grid_nx=gx)
        sim = armando_amd.Simulation(c)
        sim.time_integration(1, 5)
        sim.set_timing(True)
        sim.reset_pass_times()
        sim.time_integration(6, 20)
        us[name] = 1e3 * sim.pass_times()["reorder"][0] / 20
        sim.close()
    print(f"[gpu] reorder of 2,400 particles: {us}", flush=True)
    assert us["tall"] <= 10 * us["wide"]
