"""arm_download and arm_download_rates, the C entry points with interleaved
vectors x(dim, n), against the calls with an array per axis that Simulation
uses: every field, alone and with others, null pointers for the rest, equal bit
for bit, nothing written past a field's end.  The downloads unsort into the
inactive state's arrays: steps after them equal those of a run that was never
looked at."""
import ctypes as C
import time

import numpy as np
import pytest

import armando_amd
from armando_amd import cases

pytestmark = pytest.mark.gpu

STATE = ("x", "v", "rho", "p", "u")
RATES = ("drho", "a", "du", "av", "divv")
VECTORS = ("x", "v", "a", "av")
SETS = [(0, 1, 2, 3, 4), (0,), (1,), (2,), (3,), (4,), (1, 3), (0, 4), (2, 3, 4), ()]
GUARD = -7.25


def make(name, prec):
    if name == "2d":
        return cases.dam_break_small(scale=0.03, precision=prec)
    if name == "ghosts":
        return cases.ghost_tank(col_w=0.02, col_h=0.03, tank_w=0.05, precision=prec)
    return cases.dam_break3d_small(scale=0.06, precision=prec)


def fetch(sim, call, names, on):
    d, n = sim.dim, sim.n
    buf = {k: np.full((d * n if k in VECTORS else n) + 8, GUARD)
           for q, k in enumerate(names) if q in on}
    ptr = [buf[k].ctypes.data_as(C.POINTER(C.c_double)) if k in buf else None for k in names]
    assert getattr(sim.L, call)(sim.ctx, *ptr) == armando_amd.ARM_OK
    out = {}
    for k, b in buf.items():
        assert np.all(b[-8:] == GUARD), k
        if k in VECTORS:
            pre = "" if k == "x" else k
            for a, axis in enumerate("xyz"[:d]):
                out[pre + axis] = b[a:d * n:d]
        else:
            out[k] = b[:n]
    return out


@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
@pytest.mark.parametrize("name", ["2d", "ghosts", "3d"])
def test_interleaved_downloads(name, prec):
    c = make(name, prec)
    print(f"[gpu] downloads {name} n={c['n']} prec={prec}", flush=True)
    sim, plain = armando_amd.Simulation(c), armando_amd.Simulation(c)
    sim.time_integration(1, 3)
    plain.time_integration(1, 3)
    state, rates = sim.state(), sim.rates()
    for on in SETS:
        for call, names, ref in (("arm_download", STATE, state),
                                 ("arm_download_rates", RATES, rates)):
            for k, v in fetch(sim, call, names, on).items():
                assert np.array_equal(v, ref[k]), (call, on, k)
    sim.time_integration(4, 3)
    plain.time_integration(4, 3)
    for k, v in plain.state().items():
        assert np.array_equal(v, sim.state()[k]), k
    sim.close()
    plain.close()


@pytest.mark.parametrize("prec", [cases.FP64, cases.FP32])
@pytest.mark.parametrize("name", ["2d", "3d"])
def test_arrays_of_a_small_download(name, prec):
    """state() and rates() fetch a small state in fewer copies than fields: they
    take at most 1.1 of arm_download's five.  The arrays are the caller's own."""
    c = make(name, prec)
    sim = armando_amd.Simulation(c)
    sim.time_integration(1, 2)
    buf = {k: np.empty((sim.dim if k in VECTORS else 1) * sim.n) for k in STATE}
    ptr = [buf[k].ctypes.data_as(C.POINTER(C.c_double)) for k in STATE]

    def best(call):
        t = []
        for _ in range(200):
            t0 = time.perf_counter()
            call()
            t.append(time.perf_counter() - t0)
        return 1e6 * min(t)

    us = {"state": best(sim.state), "rates": best(sim.rates),
          "arm_download": best(lambda: sim.L.arm_download(sim.ctx, *ptr))}
    print(f"[gpu] small download {name} n={sim.n} prec={prec}: {us}", flush=True)
    for v in {**sim.state(), **sim.rates()}.values():
        assert v.flags.owndata and v.flags.writeable and v.flags.c_contiguous
    sim.close()
    assert us["state"] <= 1.1 * us["arm_download"]
    assert us["rates"] <= 1.1 * us["arm_download"]
