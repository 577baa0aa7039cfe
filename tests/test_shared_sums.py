"""Linear combinations with shared partial sums: the printed lines, evaluated in FP64,
are the matrix products they stand for."""
import re

import numpy as np
import pytest

from pylbm_amd import cases
from pylbm_amd.generator.hip import _SumBuilder, _inverse_transform, _pairs, _row_parities, _transform
from pylbm_amd.scheme import Scheme


def _evaluate(builder, lines, env):
    for text in builder.lines + ["const C %s = %s;" % ln for ln in lines]:
        name, expr = re.match(r"const C (\w+) = (.*);$", text).groups()
        assert name not in env, name
        env[name] = eval(re.sub(r"C\(([-0-9.e+]+)\)", r"(\1)", expr), {}, env)
    return np.array([env["y%d" % k] for k in range(len(lines))])


@pytest.mark.parametrize("make", [lambda: cases.lid_cavity_d2q9(8), lambda: cases.taylor_green_d3q19(4),
                                  lambda: cases.d2q5q9_vectorial(8), lambda: cases.d1q3_advection(8)])
@pytest.mark.parametrize("paired", [True, False])
def test_scheme_transforms(make, paired):
    spec = Scheme(make()).kernel_spec()
    ksym = _pairs(spec) if paired else None
    x = np.random.default_rng(2).random(spec.ns)
    env = {"x%d" % k: v for k, v in enumerate(x)}
    names = ["x%d" % k for k in range(spec.ns)]
    out = ["y%d" % k for k in range(spec.ns)]
    for mat, fn, by_rows in ((spec.M, _transform, True), (spec.invM, _inverse_transform, False)):
        sig = _row_parities(spec.M, ksym) if ksym else None
        b = _SumBuilder("s")
        got = _evaluate(b, fn(b, mat, names, out, ksym, sig), dict(env))
        ref = np.array([[float(c) for c in r] for r in mat]) @ x
        assert np.allclose(got, ref, rtol=1e-13, atol=1e-13)


@pytest.mark.parametrize("seed", range(8))
def test_random_sums(seed):
    """Sums of few variables with many common pairs, repeated and opposite ones."""
    rng = np.random.default_rng(seed)
    mat = rng.choice([-1, 0, 1, 1], size=(24, 7))
    x = rng.random(7)
    b = _SumBuilder("s")
    lines = [("y%d" % i, b.combo([(int(c), "x%d" % j) for j, c in enumerate(r)])) for i, r in enumerate(mat)]
    got = _evaluate(b, lines, {"x%d" % j: v for j, v in enumerate(x)})
    assert np.allclose(got, mat @ x, rtol=1e-13, atol=1e-13)
