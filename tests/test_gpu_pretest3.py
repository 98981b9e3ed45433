"""The 3D density pass's neighbour pre-test on the matrix cores at the sizes
where its tiling can go wrong: wavefronts and tiles of 16 that are not full,
wavefronts that run over the end of a cell row, rows with a gap of empty
cells, rows of more candidates than a word group or the staging holds, rows
of more than 96 candidates (the one-by-one walk), cells wider than 2h.

Bar.  FP64: every rate within 1e-10 of the oracle's single step (a missing or
extra neighbour moves one by about 1e-2).  FP32: the force driven by the
recorded masks equals the force of the exact walk bit for bit, so the masks
hold exactly the pairs of the exact test; the continuity sums within 1e-5 of
the FP64 oracle's scale (float rounding of sums of 60 to 300 terms)."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases
from oracle import orc

pytestmark = pytest.mark.gpu

RATES = ("drho", "ax", "ay", "az", "du", "avx", "avy", "avz")


def join(a, b, shift):
    """The particles of both lattices, b's moved along x, on one grid."""
    c = dict(a)
    for k in ("x", "y", "z", "vx", "vy", "vz", "rho", "u"):
        c[k] = np.concatenate([a[k], b[k] + (shift if k == "x" else 0.0)])
    c["n"] = c["np"] = c["x"].size
    c["ox"], c["oy"], c["oz"], c["nx"], c["ny"], c["nz"] = cases.grid_for3(
        c["x"], c["y"], c["z"], c["cell"])
    return c


def lattice(name):
    box = lambda nx, ny, nz, h=1.3: cases.box_lattice3(  # noqa: E731
        nx=nx, ny=ny, nz=nz, jitter=0.1, vel=0.1, h_fac=h, seed=nx * 7 + ny)
    if name.startswith("n"):
        return box(*map(int, name[1:].split("x")))
    if name.startswith("h"):
        return box(21, 9, 8, float(name[1:]))
    if name == "gap":  # a thin column, a slab beside and above the gap
        return join(box(3, 6, 9), box(40, 6, 5), 0.9)
    if name == "far":  # two columns in the same rows, nothing between
        return join(box(5, 7, 6), box(4, 7, 6), 1.7)
    c = dict(box(19, 8, 7))  # wide cells
    c["cell"] = 1.37 * c["cell"]
    c["ox"], c["oy"], c["oz"], c["nx"], c["ny"], c["nz"] = cases.grid_for3(
        c["x"], c["y"], c["z"], c["cell"])
    return c


@pytest.mark.parametrize("name", ["n1x1x1", "n15x1x1", "n16x1x1", "n17x1x1", "n64x1x1", "n65x1x1",
                                  "n33x5x4", "n10x9x8", "h1.0", "h1.5", "h1.8", "h2.4", "gap",
                                  "far", "wide"])
def test_pretest3(name):
    c = lattice(name)
    print(f"[gpu] 3D pre-test {name} n={c['n']}", flush=True)
    P = orc.params_from(c)
    st = orc.OracleState3(c["n"], c["np"])
    st.set(**{k: c[k] for k in ("x", "y", "z", "vx", "vy", "vz", "rho", "u")})
    orc.single_step3(P, st)
    ref = {k: st.field(k).copy() for k in RATES}

    c64 = dict(c, precision=cases.FP64)
    sim = armando_amd.Simulation(c64)
    sim.link_list()
    sim.single_step()
    g = sim.rates()
    sim.close()
    for k in RATES:
        scale = np.max(np.abs(ref[k]))
        if scale == 0.0:
            assert not np.any(g[k]), k
        else:
            assert np.max(np.abs(g[k] - ref[k])) <= 1e-10 * scale, k

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
