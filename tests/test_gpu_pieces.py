"""Pieces of a cell row that span a gap are cut at the middle of their cells:
the LDS-tiled gathers on cut pieces against the direct gathers, which visit
the same neighbours in the same order with the same arithmetic, bit for bit.

The tanks hold more particles in three cell rows than a tile has records
(592), so the rows above the free surface, with wall particles on either
side only, take the cut; one is too narrow for it, one has a lone fluid
column in the gap (the cut's two parts are uneven), one leaves a part that
still exceeds the tile (the direct path takes it)."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases

pytestmark = pytest.mark.gpu

TANKS = {"filled": dict(col_w=0.26, tank_w=0.26), "half": dict(col_w=0.26, tank_w=0.6),
         "narrow": dict(col_w=0.05, tank_w=0.05), "wide": dict(col_w=0.5, tank_w=0.5)}


def tank(name, prec, heat):
    kw = TANKS["wide" if name == "column" else name]
    c = cases.dam_break(col_h=0.02, tank_h=0.05, precision=prec, heat=heat, **kw)
    if name == "column":  # every 50th surface particle rises into the gap
        top = np.nonzero(c["y"][:c["np"]] > 0.0195)[0][::50]
        c["y"] = c["y"].copy()
        c["y"][top] += 0.012
    rng = np.random.default_rng(3)
    c["vx"] = c["vx"] + 0.1 * rng.standard_normal(c["n"])
    c["vy"] = c["vy"] + 0.1 * rng.standard_normal(c["n"])
    c["u"] = 1.0 + rng.random(c["n"])
    return c


@pytest.mark.parametrize("heat", [True, False])
@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
@pytest.mark.parametrize("name", list(TANKS) + ["column"])
def test_cut_pieces_equal_direct(name, prec, heat):
    c = tank(name, prec, heat)
    print(f"[gpu] cut pieces {name} n={c['n']} prec={prec} heat={heat}", flush=True)
    out = []
    for tiled in (True, False):
        sim = armando_amd.Simulation(c)
        sim.set_gather_path(tiled)
        sim.time_integration(1, 3)
        out.append({**sim.state(), **{"r" + k: v for k, v in sim.rates().items()}})
        sim.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
