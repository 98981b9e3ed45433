"""The seam of a grid periodic in x: the tiled 2D gathers keep the cells of the
other end in the tile of a piece that holds the first or last cell column, and
walk them after the piece's own rows, as the direct gathers do: bit for bit the
same, over runs in which particles cross the seam.

The lengths leave three cells (every cell is the seam's own or its neighbour),
one piece of both ends, two pieces that end at either, and several; the dense
one holds more than 32 candidates a row and more records than a tile."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases

pytestmark = pytest.mark.gpu

# particles along, across, h / dx
CHANNELS = {"three cells": (8, 6, 1.3), "one piece": (40, 9, 1.3), "both ends": (50, 21, 1.3),
            "two pieces": (70, 10, 1.3), "pieces": (400, 12, 1.3), "dense": (70, 30, 4.1)}


@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
@pytest.mark.parametrize("name", list(CHANNELS))
def test_seam_equals_direct(name, prec):
    ni, nj, h = CHANNELS[name]
    dx = 1e-4
    c = cases.heated_channel(length=ni * dx, width=nj * dx, dx=dx, h_fac=h, precision=prec)
    rng = np.random.default_rng(11)
    c["vx"] = c["vx"] + 0.5 * rng.standard_normal(c["n"])
    c["vy"] = c["vy"] + 0.05 * rng.standard_normal(c["n"])
    c["x"] = (c["x"] + 0.3 * dx * rng.standard_normal(c["n"])) % (ni * dx)
    print(f"[gpu] seam {name} n={c['n']} nx={c['nx']} prec={prec}", flush=True)
    out = []
    for tiled in (True, False):
        sim = armando_amd.Simulation(c)
        sim.set_gather_path(tiled)
        sim.time_integration(1, 5)
        out.append({**sim.state(), **{"r" + k: v for k, v in sim.rates().items()}})
        sim.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
