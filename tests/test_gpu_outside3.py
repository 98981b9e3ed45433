"""3D gathers on particles outside the hash grid.  arm_link_list sorts them into
cell 0 and raises ARM_ERR_DOMAIN; a program that goes on gets their pairs all
the same: 64 particles moved thousands of cells away have the rates that they
have inside.  (FP64 form: the FP32 form's upload already refuses them.)

Positions are multiples of 2^-14 and the shifts of 2^-3, held exactly: the pairs
and their terms are the same, up to the order of the sums (some 60 terms rounded
to 2^-53: 1e-12 of a field's largest value)."""
import numpy as np
import pytest

import armando_amd
from armando_amd import ArmandoError, cases

pytestmark = pytest.mark.gpu

TOL = 1e-12
RATES = ("drho", "ax", "ay", "az", "du", "avx", "avy", "avz")


def block():
    dx = 2.0 ** -7
    I = np.meshgrid(*3 * [np.arange(4)], indexing="ij")
    rng = np.random.default_rng(5)
    c = cases.box_lattice3(nx=4, ny=4, nz=4, dx=dx, vel=0.1)
    for k, a in enumerate("xyz"):
        c[a] = (I[k].ravel() + 0.5) * dx + rng.integers(-8, 9, 64) * 2.0 ** -14
    c["h"] = 1.5 * dx
    c["cell"] = 2.0 * c["h"]
    c["ox"] = c["oy"] = c["oz"] = -4.0 * c["cell"]
    c["nx"] = c["ny"] = c["nz"] = 12
    return c


def rates(c, raises):
    sim = armando_amd.Simulation(c)
    if raises:
        with pytest.raises(ArmandoError) as e:
            sim.link_list()
        assert e.value.code == -4
    else:
        sim.link_list()
    sim.single_step()
    r = sim.rates()
    sim.close()
    return r


@pytest.mark.parametrize("shift", [(64.0, 0.0, 0.0), (-32.0, -0.125, 0.0), (0.0, 32.0, 48.0)])
def test_rates_outside_the_grid(shift):
    c = block()
    ref = rates(c, False)
    far = dict(c)
    for a, d in zip("xyz", shift):
        far[a] = c[a] + d
    print(f"[gpu] outside the grid, shift {shift}", flush=True)
    got = rates(far, True)
    for k in RATES:
        d = np.max(np.abs(got[k] - ref[k]))
        assert d <= TOL * np.max(np.abs(ref[k])), (k, d)
