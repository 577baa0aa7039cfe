"""The temporally blocked runs against one launch per step, bit for bit, at the sizes
where tiles, regions and launches end."""
import numpy as np
import pytest

from pylbm_amd import Simulation, cases, demos

pytestmark = pytest.mark.gpu


def _equal(make, dtype, nsteps):
    a, b = Simulation(make(), dtype=dtype), Simulation(make(), dtype=dtype)
    assert a._blocking_shape() is not None
    b.temporal_blocking = False
    for n in nsteps:
        a.run(n)
        b.run(n)
        assert a.nt == b.nt and a.t == b.t
        for k in range(a.ns):
            assert np.isfinite(b.F[k]).all(), (n, k)
            assert np.array_equal(a.F[k], b.F[k]), (n, k)


# 1D tiles are 128 cells with a halo of up to 64: a box smaller than the halo, one tile,
# one cell more, and many tiles; a launch of 64 steps, one more, and a few
@pytest.mark.parametrize("dtype", ["float64", "float32-shifted", "float16"])
@pytest.mark.parametrize("n", [5, 64, 128, 129, 1000])
def test_1d_periodic_and_walls(hip, n, dtype):
    for walls in (False, True):
        _equal(lambda: cases.d1q3_advection(n, walls=walls), dtype, (64, 65, 3))


@pytest.mark.parametrize("n", [40, 777])
def test_1d_shock_tube(hip, n):
    _equal(lambda: demos.riemann_euler(1.0 / n)[0], "float64", (130,))
