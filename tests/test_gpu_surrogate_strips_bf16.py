"""The convolution strips on bfloat16 operands (test_conv_strips runs float16): every kind of
output at the sizes where strips and segments end, held to 2 unit roundoffs of its
one rounding, FP32 outputs to FP32 accumulation."""
import ctypes

import numpy as np
import pytest

from oracle import surrogate as osur
from test_gpu_surrogate import UNIT, _dec, _enc

pytestmark = pytest.mark.gpu
ELEM, CODE = "bfloat16", 1


def _p(x):
    return ctypes.c_void_p(x)


@pytest.mark.parametrize("N,H,W", [(1, 1, 16), (1, 5, 48), (2, 7, 96), (9, 130, 64)])
@pytest.mark.parametrize("cin,cout,epi", [(64, 32, 0), (32, 32, 0), (64, 64, 0), (32, 64, 1), (64, 32, 2), (64, 64, 2)])
def test_conv_strips_bfloat16(hip, N, H, W, cin, cout, epi):
    rng = np.random.default_rng(H + W + cin + cout)
    x, z = rng.normal(size=(N, H, W, cin)), rng.normal(size=(N, H, W, cout))
    w, b = rng.normal(0.0, 0.05, (9, cin, cout)).astype(np.float32), rng.normal(size=cout).astype(np.float32)
    out = np.empty((N, H, W, cout), np.float32 if epi == 1 else np.uint16)
    bufs = [hip.upload(w), hip.upload(b), hip.malloc(9 * cin * cout * 2), hip.upload(_enc(x, ELEM)),
            hip.upload(_enc(z, ELEM)), hip.malloc(out.nbytes)]
    ow, ob, wpk, ox, oz, oo = bufs
    hip.check(hip.lib.lbm_sur_pack(_p(ow), cin, cout, cin, cout, _p(wpk), _p(None), CODE, hip.stream), "pack")
    hip.check(hip.lib.lbm_sur_conv(_p(ox), cin, _p(wpk), _p(ob), _p(oz), _p(oo), _p(None), cout, epi, N, H, W, CODE,
                                   hip.stream), "conv")
    hip.d2h(out, oo)
    for q in bufs:
        hip.free(q)
    ref = osur.conv3x3(_dec(_enc(x, ELEM), ELEM), _dec(_enc(w, ELEM), ELEM), b.astype(np.float64) if epi < 2 else 0.0)
    if epi == 0:
        ref = osur.silu(ref)
    elif epi == 2:
        ref = ref * osur.silu_grad(_dec(_enc(z, ELEM), ELEM))
    got = out if epi == 1 else _dec(out, ELEM)
    tol = 1e-6 if epi == 1 else 2 * UNIT[ELEM]
    assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
