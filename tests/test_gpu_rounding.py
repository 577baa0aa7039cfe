"""Rounding of the generated arithmetic where it carries a format's accuracy."""
import re

import numpy as np
import pytest

from pylbm_amd import Simulation, cases
from pylbm_amd.generator.hip import (_SumBuilder, _deviation_collision_lines, _inverse_transform, _pairs,
                                     _row_parities, _transform)
from pylbm_amd.scheme import Scheme

pytestmark = pytest.mark.gpu


def _single_roundings(spec, f, omega, cref):
    """One collision of the FP32 deviations f (ns, cells) with every product and sum rounded
    on its own (numpy float32 rounds each operation), sums in the order of the rows."""
    ns, C = spec.ns, np.float32
    names = ["%s%d" % (v, k) for v in "fm" for k in range(ns)]
    fv, mv = names[:ns], names[ns:]
    ksym = _pairs(spec)
    sig = _row_parities(spec.M, ksym)
    assert sig == _row_parities(spec.invM, ksym, by_rows=False)
    b1, b2 = _SumBuilder("p", False), _SumBuilder("r", False)
    f2m = ["C %s = %s;" % ln for ln in _transform(b1, spec.M, fv, mv, ksym, sig)]
    coll, dm = _deviation_collision_lines(spec, False)
    m2f = ["C g%s = %s;" % (v[1:], e) for v, e in _inverse_transform(b2, spec.invM, dm, fv, ksym, sig, tag="d")]
    env = dict({v: f[k] for k, v in enumerate(fv)}, C=C, omega=omega, cref=cref)
    for text in b1.lines + f2m + coll + b2.lines + m2f:
        name, op, expr = re.match(r"(?:const )?(?:C )?(\w+) (\+?=) (.*);$", text).groups()
        value = eval(expr, {}, env)
        env[name] = env[name] + value if op == "+=" else value
    return np.stack([f[k] + env["g%d" % k] for k in range(ns)])


@pytest.mark.parametrize("shape", [(6, 5, 9), (64, 64, 64), (80, 97, 160)])
def test_fp32_deviations_round_every_operation(hip, shape):
    """3D FP32 deviations, one step per launch and (in the third box) two: the bits of the
    arithmetic without contraction and without sums shared between moments."""
    d = cases.taylor_green_d3q19(8)
    d["box"] = dict(zip("xyz", ([0.0, float(n)] for n in shape)), label=-1)
    d["init"] = {cases.RHO: 1.0}
    sim = Simulation(d, dtype="float32-shifted")
    rng = np.random.default_rng(3)
    for k in range(sim.ns):
        sim.F_halo[k] = sim.F_halo[k] * (1.0 + 0.05 * rng.standard_normal(sim.domain.shape_halo))
    spec = Scheme(d).kernel_spec()
    omega = np.array(sim.params.omega[:sim.ns], dtype=np.float32)
    cref = np.array(sim.params.cref[:sim.ns], dtype=np.float32)
    inner = (slice(None),) + (slice(1, -1),) * 3
    f = sim.container.F.fields_raw()[inner].astype(np.float32)
    for steps in (1, 2):
        sim.run(steps)
        for _ in range(steps):
            pulled = np.stack([np.roll(f[k], spec.velocities[k], axis=(0, 1, 2)) for k in range(sim.ns)])
            f = _single_roundings(spec, pulled.reshape(sim.ns, -1), omega, cref).reshape(f.shape)
        assert np.array_equal(sim.container.F.fields_raw()[inner], f)
