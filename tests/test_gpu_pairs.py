"""3D runs that advance two steps per launch give the bits of one_time_step: outer, mid and
inner extents that leave remainders of the tiles and of the planes per workgroup, odd
numbers of steps, each storage format the kernel takes, folded bounce-back copies,
source terms, and the grids on either side of the rule."""
import numpy as np
import pytest

from pylbm_amd import Simulation, bc, cases
from pylbm_amd.elements import Sphere

pytestmark = pytest.mark.gpu
FORCE = 1e-5


def _flow(shape, walls, source):
    box = dict(zip("xyz", ([0.0, float(n)] for n in shape)))
    box["label"] = [-1, -1, 0, 0, 0, 0] if walls else -1
    d = {"box": box, "space_step": 1.0, "scheme_velocity": 1, "generator": "hip",
         "schemes": [cases.d3q19_mrt(1.9, source_qx=cases.RHO * FORCE if source else None)], "init": {cases.RHO: 1.0}}
    if walls:
        d["elements"] = [Sphere([0.4 * shape[0], 0.5 * shape[1], 0.45 * shape[2]], 7.3, label=0)]
        d["boundary_conditions"] = {0: {"method": {0: bc.BounceBack}}}
    return d


def _start(d, dtype, shape):
    sim = Simulation(d, dtype=dtype)
    rng = np.random.default_rng(sum(shape))
    sim.m_halo[cases.RHO] = 1.0 + 0.01 * rng.standard_normal(sim.domain.shape_halo)
    for q in (cases.QX, cases.QY, cases.QZ):
        sim.m_halo[q] = 0.02 * rng.standard_normal(sim.domain.shape_halo)
    sim.equilibrium()
    sim.m2f()
    sim.sync()
    return sim


@pytest.mark.parametrize("shape,dtype,walls,source,paired", [
    ((77, 190, 93), "float64", False, False, True),     # rows of 16, columns of 32 and planes with a remainder
    ((97, 130, 159), "float32", False, False, True),
    ((80, 97, 160), "float32-shifted", False, True, True),
    ((77, 190, 93), "float64", True, True, True),
    ((77, 190, 93), "float32", True, False, True),
    ((160, 97, 127), "float32-shifted", True, True, True),
    ((40, 33, 32), "float64", False, False, False),     # small: one step at a time is faster
    ((40, 300, 31), "float32", False, False, False),    # narrower than a tile
    ((64, 64, 70), "float16", False, False, False),     # a format of single steps
])
@pytest.mark.parametrize("steps", [2, 5])
def test_pairs_equal_single_steps(hip, shape, dtype, walls, source, paired, steps):
    d = _flow(shape, walls, source)
    ref, sim, plain = (_start(d, dtype, shape) for _ in range(3))
    for _ in range(steps):
        ref.one_time_step()
    first = sim.container.F.ptr
    sim.run(steps)
    launches = steps // 2 + steps % 2 if paired else steps
    assert (sim.container.F.ptr != first) == (launches % 2 == 1)   # F and Fnew change places per launch
    plain.temporal_blocking = False
    plain.run(steps)
    assert sim.t == ref.t and sim.nt == ref.nt
    for k in range(sim.ns):
        want = ref.F[k]
        assert np.array_equal(sim.F[k], want)
        assert np.array_equal(plain.F[k], want)


def test_pairs_population_planes(hip):
    """The other arrangement of the populations (one array each) takes the same pairs."""
    shape = (80, 97, 160)
    d = _flow(shape, False, False)
    sims = [Simulation(d, dtype="float32", layout=lay) for lay in ("interleaved", "planes")]
    rng = np.random.default_rng(4)
    noise = 0.05 * rng.standard_normal((sims[0].ns,) + tuple(sims[0].domain.shape_halo))
    for sim in sims:
        for k in range(sim.ns):
            sim.F_halo[k] = sim.F_halo[k] * (1.0 + noise[k])
        first = sim.container.F.ptr
        sim.run(6)
        assert sim.container.F.ptr != first   # three launches
    for k in range(sims[0].ns):
        assert np.array_equal(sims[0].F[k], sims[1].F[k])
