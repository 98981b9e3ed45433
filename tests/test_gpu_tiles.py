"""2D gathers whose pieces fill their tiles: on a lattice with h = 1.7 or 1.8 dx the
cell rows hold three or four particle rows each, and a piece of a thinner one
needs up to 600 records (FP64) or 640 (FP32).  Tiled equals direct bit for bit,
reads past a full tile's last row included; and such a tile does not fall back to
the direct path: the FP64 force pass at h = 1.8 dx takes less than at 1.85, which
has more neighbours (165 and 197 us for 350,000 particles; 197 and 196 with tiles
of 592 records)."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases

pytestmark = pytest.mark.gpu

FLAGS = {"heat": None, "plain": cases.AV_VEL, "visc": cases.VISC | cases.AV_VEL}


def box(h, prec, nx=300, ny=60, **kw):
    c = cases.box_lattice(nx=nx, ny=ny, dx=0.01, jitter=0.02, precision=prec, vel=0.01, h_fac=h)
    c.update(dt=1e-7, **kw)
    return c


@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
@pytest.mark.parametrize("flags", list(FLAGS))
@pytest.mark.parametrize("h", [1.65, 1.7, 1.74, 1.8, 1.82])
def test_full_tiles_equal_direct(h, flags, prec):
    c = box(h, prec, visc_eta=1e-3)
    if FLAGS[flags] is not None:
        c["flags"] = FLAGS[flags]
    print(f"[gpu] full tiles h={h} {flags} prec={prec} n={c['n']}", flush=True)
    out = []
    for tiled in (True, False):
        sim = armando_amd.Simulation(c)
        sim.set_gather_path(tiled)
        sim.link_list()
        sim.single_step()
        r = dict(sim.rates())
        sim.time_integration(1, 2)
        out.append({**sim.state(), **{"r" + k: v for k, v in r.items()}})
        sim.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k


def test_full_tiles_do_not_fall_back():
    us = {}
    for h in (1.8, 1.85):
        sim = armando_amd.Simulation(box(h, cases.FP64, nx=700, ny=500))
        sim.time_integration(1, 5)
        sim.set_timing(True)
        sim.reset_pass_times()
        sim.time_integration(6, 40)
        us[h] = 1e3 * sim.pass_times()["force"][0] / 40
        sim.close()
    print(f"[gpu] force pass, us by h: {us}", flush=True)
    assert us[1.8] <= 0.95 * us[1.85]
