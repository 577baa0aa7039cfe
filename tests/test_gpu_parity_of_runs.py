"""The buffer that holds the state after lbm_gen_run / lbm_gen_run_blocked, called as a C
program calls them: d_f after an even number of steps and d_fnew after an odd one, whatever
the number of steps per launch, or with launch_parity the one that *parity names."""
import ctypes
import functools

import numpy as np
import pytest

from pylbm_amd import Simulation, cases

pytestmark = pytest.mark.gpu


def _state(arr):
    inner = (slice(None),) + tuple(slice(h, n - h) for n, h in zip(arr.layout.n[3 - arr.layout.dim:],
                                                                   arr.layout.halo[3 - arr.layout.dim:]))
    return arr.fields_raw()[inner]


def _check(sim, ref, nsteps, run, launches):
    for _ in range(nsteps):
        ref.one_time_step()
    c = sim.container
    parity = ctypes.c_int(7)
    sim.params.t = 0.0
    sim.rt.check(run(ctypes.byref(parity)), "run")
    sim.sync()
    free = sim.params.launch_parity
    assert parity.value == (launches if free else nsteps) % 2
    assert np.array_equal(_state((c.F, c.Fnew)[parity.value]), _state(ref.container.F))


def _box():
    d = cases.taylor_green_d3q19(8)
    d["box"] = {"x": [0.0, 80.0], "y": [0.0, 97.0], "z": [0.0, 160.0], "label": -1}   # runs in pairs
    d["init"] = {cases.RHO: 1.0}
    return d


MAKE = {"3d": (_box, "float32"), "2d": (lambda: cases.decaying_d2q9(48), "float64")}


@functools.lru_cache(maxsize=None)
def _rough(which):
    make, dtype = MAKE[which]
    sim = Simulation(make(), dtype=dtype)
    rng = np.random.default_rng(11)
    for k in range(sim.ns):
        sim.F_halo[k] = sim.F_halo[k] * (1.0 + 0.05 * rng.standard_normal(sim.domain.shape_halo))
    return sim


def _pair(which):
    out = []
    for _ in range(2):
        make, dtype = MAKE[which]
        sim = Simulation(make(), dtype=dtype)
        sim.container.F.copy_from(_rough(which).container.F)
        out.append(sim)
    return out


@pytest.mark.parametrize("free", [0, 1])
@pytest.mark.parametrize("nsteps", [0, 1, 2, 3, 4, 5, 6, 7])
def test_run(hip, nsteps, free):
    sim, ref = _pair("3d")
    sim.params.launch_parity = free
    c = sim.container
    _check(sim, ref, nsteps, lambda parity: sim.module.lbm_gen_run(
        ctypes.c_void_p(c.F.ptr), ctypes.c_void_p(c.Fnew.ptr), ctypes.byref(c.F.layout), ctypes.byref(sim.vel),
        ctypes.byref(sim.params), None, 0, nsteps, 0, 1, parity, sim.rt.stream), nsteps // 2 + nsteps % 2)


@pytest.mark.parametrize("free", [0, 1])
@pytest.mark.parametrize("nsteps", [1, 2, 5, 6, 7, 12, 13, 18])
def test_run_blocked(hip, nsteps, free):
    sim, ref = _pair("2d")
    sim.params.launch_parity = free
    c = sim.container
    _check(sim, ref, nsteps, lambda parity: sim.module.lbm_gen_run_blocked(
        ctypes.c_void_p(c.F.ptr), ctypes.c_void_p(c.Fnew.ptr), ctypes.byref(c.F.layout), ctypes.byref(sim.params),
        nsteps, 6, 16, 16, parity, sim.rt.stream), -(-nsteps // 6))
