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


def _stripes(n, valued):
    """Fluid columns one cell wide between solid ones: three links per cell, more than
    the link list of a region holds (every wall carries the lid's value when valued)."""
    from pylbm_amd.elements import Parallelogram
    d = cases.lid_cavity_d2q9(n)
    d["elements"] = [Parallelogram((x - 0.25, -1.0), (0.5, 0.0), (0.0, n + 2.0), label=1 if valued else 0)
                     for x in np.arange(0.5, n, 2.0)]
    return d


# regions with more links than their list holds, with and without table entries, and
# lists longer than one link per thread (every wall of a small box, wrapped many times
# into the region)
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_2d_dense_and_long_link_lists(hip, dtype):
    for valued in (False, True):
        _equal(lambda: _stripes(48, valued), dtype, (9,))

    def small():
        d = cases.lid_cavity_d2q9(9)
        d["box"]["label"] = [1, 1, 1, 1]
        return d
    _equal(small, dtype, (13,))
    _equal(lambda: cases.with_bouzidi(cases.karman_d2q9(90, 50, radius=9.3, center=(25.2, 24.7))), dtype, (14,))


# ragged 2D boxes: tiles and regions that do not divide them, boxes thinner than a tile,
# and (more than 256 tiles in half planes) two workgroups per CU
@pytest.mark.parametrize("dtype", ["float64", "float32", "bfloat16"])
@pytest.mark.parametrize("nx,ny", [(4, 300), (301, 5), (37, 41), (700, 611)])
def test_2d_ragged(hip, nx, ny, dtype):
    _equal(lambda: cases.forced_periodic_d2q9(nx=nx, ny=ny, g0=1e-7), dtype, (25, 2))
