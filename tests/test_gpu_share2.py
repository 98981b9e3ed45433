"""The 2D adjoint's gathers deal a particle's neighbours to one, two or four
wavefronts, by the number of particles.  A block far from every other one gets
the same gradient whatever that number: it is differentiated alone and beside
enough copies of itself to reach each form.

The forms differ in the order of the sums over about 21 pairs, each rounded to
2^-53 (FP64) or 2^-24 (FP32) of terms up to some hundred times the sum; the
copies' positions, shifted by whole cells, are rounded to 2^-53 of the domain's
length, 1e4 spacings.  Bound: 1e-9 and 5e-4 of the largest component."""
import numpy as np
import pytest

import armando_amd
from armando_amd import cases

pytestmark = pytest.mark.gpu

TOL = {cases.FP64: 1e-9, cases.FP32: 5e-4}


def gradient(prec, copies, flags):
    b = cases.box_lattice(nx=40, ny=36, dx=0.01, jitter=0.1, precision=prec, vel=0.5)
    pitch = 20  # cells; the block spans 15.4
    c = dict(b)
    for k in ("x", "y", "vx", "vy", "rho", "u"):
        c[k] = np.concatenate([b[k] + (q * pitch * b["cell"] if k == "x" else 0.0)
                               for q in range(copies)])
    c["n"] = c["np"] = b["n"] * copies
    c["nx"] = b["nx"] + pitch * (copies - 1)
    c["flags"] = b["flags"] | flags
    c["visc_eta"] = 0.05
    print(f"[gpu] share2 n={c['n']} prec={prec} flags={flags}", flush=True)
    sim = armando_amd.Simulation(c)
    J, da, g, _ = sim.adjoint_rollout(4, 2, np.arange(0, b["n"], 3, dtype=np.int32))
    sim.close()
    return J, da, g[:b["n"]]


@pytest.mark.parametrize("flags", [0, cases.VISC])
@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
def test_forms_agree(prec, flags):
    ref = gradient(prec, 1, flags)
    assert np.max(np.abs(ref[2])) > 0
    for copies in (40, 70):  # of 1,440 particles: two wavefronts, one
        for got, want in zip(gradient(prec, copies, flags), ref):
            d = np.max(np.abs(np.asarray(got) - want))
            assert d <= TOL[prec] * np.max(np.abs(want)), (copies, d)
