"""Population stores into the caches (24 to 320 MB of populations): layouts whose strides
reach past 4 GiB, and FP64 against the oracle."""
import ctypes

import numpy as np
import pytest

from conftest import rel_err
from oracle.lbm import Simulation as Oracle
from pylbm_amd import Simulation, cases
from pylbm_amd.runtime import LbmLayout

pytestmark = pytest.mark.gpu


def _box(shape):
    d = cases.taylor_green_d3q19(8)
    d["box"] = dict(zip("xyz", ([0.0, float(n)] for n in shape)), label=-1)
    return d


def _copy_populations(rt, ns, es, src, src_lay, dst, dst_lay):
    size = src_lay.n[0] * src_lay.n[1] * src_lay.pitch * es
    for k in range(ns):
        rt.d2d(dst + k * dst_lay.pop_stride * es, src + k * src_lay.pop_stride * es, size)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("fold", [1, 0])
def test_strides_past_4_gib(hip, dtype, fold):
    """19 populations 2^32 / 15 bytes apart: fewer than 2^31 elements, byte offsets past 2^32."""
    d = _box((64, 62, 70))
    d["init"] = {cases.RHO: 1.0}
    sim = Simulation(d, dtype=dtype, layout="planes")
    rng = np.random.default_rng(5)
    for k in range(sim.ns):
        sim.F_halo[k] = sim.F_halo[k] * (1.0 + 0.05 * rng.standard_normal(sim.domain.shape_halo))
    F, rt = sim.container.F, sim.rt
    L, es = F.layout, F.layout.elem_size
    wide = LbmLayout.from_buffer_copy(L)
    wide.pop_stride = 2 ** 32 // 15 // es // 64 * 64
    nbytes = sim.ns * wide.pop_stride * es
    assert nbytes > 2 ** 32 and nbytes // es < 2 ** 31
    a = rt.malloc(nbytes)
    b = rt.malloc(nbytes)
    try:
        _copy_populations(rt, sim.ns, es, F.ptr, L, a, wide)
        step = lambda f, fn, lay: rt.check(sim.module.lbm_gen_step(   # noqa: E731
            ctypes.c_void_p(f), ctypes.c_void_p(fn), ctypes.byref(lay), ctypes.byref(sim.params), fold, rt.stream), "step")
        step(F.ptr, sim.container.Fnew.ptr, L)
        step(a, b, wide)
        _copy_populations(rt, sim.ns, es, b, wide, F.ptr, L)
        inner = (slice(None),) + (slice(1, -1),) * 3
        assert np.array_equal(F.fields_raw()[inner], sim.container.Fnew.fields_raw()[inner])
    finally:
        rt.sync()
        rt.free(a)
        rt.free(b)


@pytest.mark.parametrize("shape", [(48, 45, 50), (50, 49, 65)])
def test_fp64_against_the_oracle(hip, shape):
    """39 and 62 MB: one step per call, each value within a few roundings of the oracle's."""
    d = _box(shape)
    sim, ref = Simulation(d, dtype="float64"), Oracle(d)
    for _ in range(2):
        sim.one_time_step()
        ref.one_time_step()
    for s in (cases.RHO, cases.QX, cases.QY, cases.QZ):
        assert rel_err(sim.m[s], ref.m(s)) <= 1e-12
