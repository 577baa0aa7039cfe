"""Two steps per launch where their difference matters: source terms in X, Y, Z and t (wrapped
coordinates, each step's own t), other stencils than D3Q19 (other populations per plane of
LDS, pulls along all three diagonals), and a kernel that does not fit its registers."""
import numpy as np
import pytest
import sympy as sp

from pylbm_amd import Simulation, bc, cases, demos
from pylbm_amd.elements import Sphere

pytestmark = pytest.mark.gpu
X, Y, Z, T = sp.symbols("X Y Z t")
LINEAR = cases.RHO * 1e-5 * (1 + 0.02 * X - 0.03 * Y + 0.01 * Z) * (1 + 0.1 * T)
WAVES = cases.RHO * 1e-5 * sp.sin(0.1 * X + 0.02 * Y - 0.05 * Z) * sp.cos(0.3 * T)


def _d3q15():
    x, y, z = sp.symbols("X Y Z")
    r, qx, qy, qz = cases.RHO, cases.QX, cases.QY, cases.QZ
    n = x ** 2 + y ** 2 + z ** 2
    c = sp.Rational(7, 3)
    return {"velocities": list(range(7)) + list(range(19, 27)), "conserved_moments": [r, qx, qy, qz],
            "polynomials": [1, x, y, z, n, x ** 2 - y ** 2, y ** 2 - z ** 2, x * y, y * z, x * z, x * n, y * n, z * n,
                            x * y * z, n ** 2],
            "equilibrium": [r, qx, qy, qz, r + qx ** 2 + qy ** 2 + qz ** 2, qx ** 2 - qy ** 2, qy ** 2 - qz ** 2,
                            qx * qy, qy * qz, qx * qz, c * qx, c * qy, c * qz, 0, c * r],
            "relaxation_parameters": [0] * 4 + [1.2] + [1.6] * 5 + [1.1] * 3 + [1.3] * 2}


def _box(shape, scheme, walls):
    d = {"box": dict(zip("xyz", ([0.0, float(n)] for n in shape)), label=[-1, -1, 0, 0, 0, 0] if walls else -1),
         "space_step": 1.0, "scheme_velocity": 1, "generator": "hip", "schemes": [scheme], "init": {cases.RHO: 1.0}}
    if walls:
        d["elements"] = [Sphere([0.4 * shape[0], 0.5 * shape[1], 0.45 * shape[2]], 7.3, label=0)]
        d["boundary_conditions"] = {0: {"method": {0: bc.BounceBack}}}
    return d


def _state(sim):
    return sim.container.F.fields_raw()[(slice(None),) + (slice(1, -1),) * 3]


def _same_bits(d, dtype, steps, launches):
    ref, sim = Simulation(d, dtype=dtype), Simulation(d, dtype=dtype)
    rng = np.random.default_rng(12)
    for c in ref.scheme.consm:   # rough conserved moments, and with the sources' first step off equilibrium
        ref.m_halo[c] = ref.m_halo[c] + 0.02 * rng.standard_normal(ref.domain.shape_halo)
    ref.equilibrium()
    ref.m2f()
    ref.sync()
    sim.container.F.copy_from(ref.container.F)
    for _ in range(steps):
        ref.one_time_step()
    first = sim.container.F.ptr
    sim.run(steps)
    assert (sim.container.F.ptr != first) == (launches % 2 == 1)
    assert sim.t == ref.t
    want = _state(ref)
    assert np.isfinite(want).all()
    assert np.array_equal(_state(sim), want)


@pytest.mark.parametrize("shape,dtype,walls", [((97, 130, 159), "float32", False), ((77, 190, 93), "float64", False),
                                               ((80, 97, 160), "float32-shifted", True), ((77, 190, 93), "float64", True)])
def test_linear_source(hip, shape, dtype, walls):
    _same_bits(_box(shape, cases.d3q19_mrt(1.9, source_qx=LINEAR), walls), dtype, 5, 3)


@pytest.mark.parametrize("dtype,launches", [("float32", 3), ("float64", 5)])
def test_source_of_waves(hip, dtype, launches):
    """In FP64 the two-step kernel of this source spills registers: five single steps."""
    _same_bits(_box((97, 130, 159), cases.d3q19_mrt(1.9, source_qx=WAVES), False), dtype, 5, launches)


@pytest.mark.parametrize("shape,dtype,walls", [((97, 130, 159), "float32", False), ((77, 190, 93), "float64", False),
                                               ((97, 130, 159), "float64", True)])
def test_d3q15(hip, shape, dtype, walls):
    _same_bits(_box(shape, _d3q15(), walls), dtype, 5, 3)


@pytest.mark.parametrize("dtype", ["float32", "float64", "float32-shifted"])
def test_d3q6(hip, dtype):
    d = demos.advection_3d(1 / 97)[0]
    _same_bits(d, dtype, 5, 3)
