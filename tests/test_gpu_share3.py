"""The 3D gathers deal a particle's candidates to one, two, four or eight
wavefronts, by the number of particles.  A block of particles far from every
other one must get the same results whatever that number: it is stepped alone
and beside enough copies of itself to reach each form, and its state, rates and
gradients compared.

The forms differ in the order of the sums over about 75 pairs, each rounded to
2^-53 (FP64) or 2^-24 (FP32) of terms up to some hundred times the sum; the
copies' positions, shifted by whole cells, are rounded to 2^-53 of the domain's
length, 1e4 spacings.  Bound: 1e-9 and 5e-4 of a field's largest value."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases

pytestmark = pytest.mark.gpu

TOL = {cases.FP64: 1e-9, cases.FP32: 5e-4}
COPIES = (12, 20, 40, 60)  # of 2,548 particles: 8/4/2/1 wavefronts in FP32, 4/2/1/1 in FP64


def blocks(prec, copies):
    b = cases.box_lattice3(nx=14, ny=14, nz=13, precision=prec, vel=0.5)
    pitch = 10  # cells; the block spans 5.4
    c = dict(b)
    for k in ("x", "y", "z", "vx", "vy", "vz", "rho", "u"):
        c[k] = np.concatenate([b[k] + (q * pitch * b["cell"] if k == "x" else 0.0)
                               for q in range(copies)])
    c["n"] = c["np"] = b["n"] * copies
    c["nx"] = b["nx"] + pitch * (copies - 1)
    return c, b["n"]


def step(prec, copies):
    c, n = blocks(prec, copies)
    print(f"[gpu] share3 n={c['n']} prec={prec}", flush=True)
    sim = armando_amd.Simulation(c)
    sim.time_integration(1, 3)
    out = {**sim.state(), **{"r" + k: v for k, v in sim.rates().items()}}
    sim.close()
    sim = armando_amd.Simulation(c)
    out["J"], out["da"], out["g"], _ = sim.adjoint_rollout(4, 2, np.arange(0, n, 3, dtype=np.int32))
    sim.close()
    first = {k: (v if np.ndim(v) == 0 else v[:n]) for k, v in out.items()}
    return first, {k: v[-n:] for k, v in out.items() if np.ndim(v) and k not in ("x", "g")}


@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
def test_forms_agree(prec):
    ref, _ = step(prec, 1)
    for copies in COPIES:
        first, last = step(prec, copies)
        for got in (first, last):
            for k, v in got.items():
                d = np.max(np.abs(np.asarray(v) - ref[k]))
                assert d <= TOL[prec] * np.max(np.abs(ref[k])), (copies, k, d)
