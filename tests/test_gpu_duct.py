"""3D boxes with inflow values and outflow copies fold into the step with a table on two
faces (batches of entries, planes taken from both ends): the bits of the link launches,
for extents with an even and an odd number of planes and a single plane between the faces.
Stores into the caches (24 to 320 MB of populations) give the bits of stores past them."""
import numpy as np
import pytest

from pylbm_amd import Simulation, bc, cases

pytestmark = pytest.mark.gpu


def _inflow(f, m, x, y, z):
    m[cases.RHO], m[cases.QX], m[cases.QY], m[cases.QZ] = 1.0, 0.05 + 0.01 * np.sin(y + z), 0.0, 0.01


def _duct(shape, axis):
    label = [0] * 6
    label[2 * axis:2 * axis + 2] = [1, 2]
    box = dict(zip("xyz", ([0.0, float(n)] for n in shape)), label=label)
    outflow = (bc.NeumannX, bc.NeumannY, bc.NeumannZ)[axis]
    return {"box": box, "space_step": 1.0, "scheme_velocity": 1, "generator": "hip",
            "schemes": [cases.d3q19_mrt(1.9)], "init": {cases.RHO: 1.0},
            "boundary_conditions": {0: {"method": {0: bc.BounceBack}},
                                    1: {"method": {0: bc.AntiBounceBack}, "value": _inflow},
                                    2: {"method": {0: outflow}}}}


def _noise(sim):
    rng = np.random.default_rng(7)
    for k in range(sim.ns):
        sim.F_halo[k] = sim.F_halo[k] * (1.0 + 0.05 * rng.standard_normal(sim.domain.shape_halo))
    sim.container.Fnew.copy_from(sim.container.F)


@pytest.mark.parametrize("shape,axis", [((24, 13, 17), 0), ((25, 40, 9), 0), ((3, 16, 16), 0), ((12, 9, 70), 1),
                                        ((11, 14, 66), 2)])
@pytest.mark.parametrize("dtype", ["float64", "float32", "float32-shifted", "float16"])
def test_duct_fold_equals_launches(hip, shape, axis, dtype):
    d = _duct(shape, axis)
    a, b = Simulation(d, dtype=dtype), Simulation(d, dtype=dtype, initialize=False)
    assert a._wrap and a.params.bbtab_bits
    b.fold_links = False
    b._initialize()
    assert not b._wrap
    for sim in (a, b):
        _noise(sim)
        sim.one_time_step()
        sim.run(7)
    for k in range(a.ns):
        assert np.array_equal(a.F[k], b.F[k]), k


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
def test_cached_stores(hip, dtype):
    d = cases.taylor_green_d3q19(96)   # 269 MB in FP64: past / into the caches by format
    a, b = Simulation(d, dtype=dtype), Simulation(d, dtype=dtype)
    b.params.vec_cells = 4             # four cells per thread, always past the caches
    for sim in (a, b):
        sim.run(3)
        sim.one_time_step()
    for k in range(a.ns):
        assert np.array_equal(a.F[k], b.F[k]), k
