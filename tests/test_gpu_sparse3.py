"""The 3D density pass where a wavefront's particles lie in many cell rows (spray,
thin sheets, narrow channels, beside dense fluid): there the lanes make the
neighbour test themselves instead of the sweeps on the matrix cores.

Bar, as for the sweeps.  FP64: every rate within 1e-10 of the oracle's single
step.  FP32: the force driven by the recorded masks equals the force of the exact
walk bit for bit; the continuity sums within 1e-5 of the FP64 oracle's scale.
And cost: the density pass of thin spray takes at most three times its force
pass (1.6 as measured; ten times when every row was swept)."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases
from oracle import orc

pytestmark = pytest.mark.gpu

RATES = ("drho", "ax", "ay", "az", "du", "avx", "avy", "avz")


def particles(x, y, z, seed):
    """Particles at given places, with the lattice case's constants."""
    c, r = cases.box_lattice3(nx=2, ny=2, nz=2), np.random.default_rng(seed)
    n = x.size
    c.update(n=n, np=n, x=x, y=y, z=z, rho=1000.0 * (1 + 0.01 * r.uniform(-1, 1, n)),
             u=1.0 + 0.5 * r.random(n), **{"v" + a: 0.1 * r.uniform(-1, 1, n) for a in "xyz"})
    c["ox"], c["oy"], c["oz"], c["nx"], c["ny"], c["nz"] = cases.grid_for3(x, y, z, c["cell"])
    return c


def spray(n, per_cell, seed=3):
    cell = cases.box_lattice3(nx=2, ny=2, nz=2)["cell"]
    p = np.random.default_rng(seed).random((n, 3)) * (n / per_cell) ** (1 / 3) * cell
    return particles(*(np.ascontiguousarray(a) for a in p.T), seed)


def make(name):
    if name.startswith("spray"):
        n, per_cell = name[5:].split("@")
        return spray(int(n), float(per_cell))
    if name.startswith("n"):
        nx, ny, nz = map(int, name[1:].split("x"))
        return cases.box_lattice3(nx=nx, ny=ny, nz=nz, jitter=0.1, vel=0.1, seed=nx * 7 + ny)
    a, b = cases.box_lattice3(nx=20, ny=18, nz=16), spray(3000, 0.5)  # a block in spray
    keep = ~((b["x"] < 0.22) & (b["y"] < 0.2) & (b["z"] < 0.18))
    return particles(*(np.concatenate([a[k], b[k][keep]]) for k in "xyz"), 5)


@pytest.mark.parametrize("name", ["spray1@1", "spray70@0.3", "spray3000@0.3", "spray3000@1",
                                  "spray3000@3", "spray3000@8", "spray140000@0.3", "n1x40x40",
                                  "n2x40x40", "n3x30x30", "n4x30x30", "n30x30x2", "n3x3x300",
                                  "mixed"])
def test_sparse3(name):
    c = make(name)
    print(f"[gpu] sparse 3D {name} n={c['n']}", flush=True)
    P = orc.params_from(c)
    st = orc.OracleState3(c["n"], c["np"])
    st.set(**{k: c[k] for k in ("x", "y", "z", "vx", "vy", "vz", "rho", "u")})
    orc.single_step3(P, st)
    ref = {k: st.field(k).copy() for k in RATES}
    sim = armando_amd.Simulation(dict(c, precision=cases.FP64))
    sim.link_list()
    sim.single_step()
    g = sim.rates()
    sim.close()
    for k in RATES:
        assert np.max(np.abs(g[k] - ref[k])) <= 1e-10 * np.max(np.abs(ref[k])), k
    c32 = dict(c, precision=cases.FP32)
    got = []
    for drop in (False, True):  # masks kept, or dropped by a second link_list
        sim = armando_amd.Simulation(c32)
        sim.link_list()
        sim.density(0)
        if drop:
            sim.link_list()
        sim.eos()
        sim.internal_force(c32["flags"])
        got.append(sim.rates())
        sim.close()
    for k in ("ax", "ay", "az", "du"):
        assert np.array_equal(got[0][k], got[1][k]), k
    assert np.max(np.abs(got[0]["drho"] - ref["drho"])) <= 1e-5 * max(np.max(np.abs(ref["drho"])), 1e-30)


@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
def test_cost_of_spray(prec):
    c = dict(spray(200000, 0.3), precision=prec, dt=1e-8)
    sim = armando_amd.Simulation(c)
    sim.time_integration(1, 5)
    sim.set_timing(True)
    sim.reset_pass_times()
    sim.time_integration(6, 20)
    us = {k: 1e3 * ms / 20 for k, (ms, _) in sim.pass_times().items()}
    sim.close()
    print(f"[gpu] spray prec={prec}: density {us['density']:.1f} us, force {us['force']:.1f}", flush=True)
    assert us["density"] <= 3 * us["force"]
