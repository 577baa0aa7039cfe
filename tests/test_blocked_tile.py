"""The tile rule of the temporally blocked 2D runs (CPU): every shape it returns fits the
kernel, short runs get shapes of their own length, and single steps stay where they are faster."""
import itertools

import pytest

from pylbm_amd.simulation import _blocked_tile


@pytest.mark.parametrize("ns,es", [(9, 8), (9, 4), (9, 2), (14, 8), (4, 4), (1, 4), (40, 8)])
def test_shapes_fit(ns, es):
    plane = min((160 * 1024) // (2 * ns * es + 12), 65528 // ((ns - 1) * es) if ns > 1 else 1 << 30)
    for n0, n1, links, nsteps in itertools.product((2, 7, 64, 333, 3000), (5, 128, 1000), (False, True), (2, 3, 7, 13, 32)):
        shape = _blocked_tile(ns, es, n0, n1, links, nsteps)
        if shape is None:
            continue
        nt, tm, ti = shape
        assert 2 <= nt <= min(n0, n1, nsteps) and 1 <= tm <= n0 and 1 <= ti <= n1
        assert (tm + 2 * nt) * (ti + 2 * nt) <= plane


def test_short_runs():
    """1000^2 FP32: two steps one at a time, and seven steps not with the tile of long runs (12.4 us
    per step with it, 10.5 with 6 of 32 x 32 and a single one, 8.6 with this rule)."""
    assert _blocked_tile(9, 4, 1000, 1000, False, 2) is None
    assert _blocked_tile(9, 4, 256, 256, False, 2) is not None
    for nsteps in (3, 5, 7, 9, 13):
        nt = _blocked_tile(9, 4, 1000, 1000, False, nsteps)[0]
        launches = -(-nsteps // nt)
        assert nt == -(-nsteps // launches)   # no launch is shorter than the tile was chosen for by more than one


def test_fp64_of_many_populations():
    """D2Q9 + D2Q5 FP64: regions of half the LDS on large grids (1000^2 35.3 us per step with
    4 steps of 16 x 16, 30.3 with 3 of 8 x 16)."""
    nt, tm, ti = _blocked_tile(14, 8, 1000, 1000, False, 32)
    assert (tm + 2 * nt) * (ti + 2 * nt) <= (80 * 1024) // (2 * 14 * 8 + 12)
