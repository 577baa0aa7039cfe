"""The surrogate's weight gradient, convolution strips and one-launch Adam step at the
sizes where segments, strips and workgroups end.

The device's 16-bit operands are given, so a weight gradient differs from the FP64 sum of
the same products only by FP32 accumulation: at most K roundings of 2^-24 on a random
walk, 1e-5 in the relative 2-norm for the K = 8320 pixels here.  A convolution output
is rounded once to 16 bits (unit roundoff u), held to 2 u."""
import ctypes

import numpy as np
import pytest

from oracle import surrogate as osur
from test_gpu_surrogate import UNIT, _dec, _enc

pytestmark = pytest.mark.gpu
CODE = {"float16": 0, "bfloat16": 1}


def _p(x):
    return ctypes.c_void_p(x)


# H = 1 with more segments than workgroups, odd H, a last segment of 32 pixels, strips
# that do not divide H
@pytest.mark.parametrize("N,H,W", [(260, 1, 32), (1, 5, 32), (2, 7, 96), (3, 37, 64)])
@pytest.mark.parametrize("cin,cout", [(64, 32), (32, 32), (32, 64), (64, 64)])
@pytest.mark.parametrize("elem", ["float16", "bfloat16"])
def test_wgrad_strips(hip, N, H, W, cin, cout, elem):
    rng = np.random.default_rng(N * 1000 + H + cin + cout)
    x, dz = rng.normal(size=(N, H, W, cin)), rng.normal(size=(N, H, W, cout))
    nblk = hip.lib.lbm_sur_wgrad_blocks()
    bufs = [hip.upload(_enc(x, elem)), hip.upload(_enc(dz, elem)), hip.malloc(nblk * (9 * cin * cout + cout) * 4),
            hip.malloc(9 * cin * cout * 4), hip.malloc(cout * 4)]
    hip.check(hip.lib.lbm_sur_wgrad(_p(bufs[0]), cin, _p(bufs[1]), cout, N, H, W, _p(bufs[2]), _p(bufs[3]), _p(bufs[4]),
                                    CODE[elem], hip.stream), "wgrad")
    dw, db = np.empty((9, cout, cin), np.float32), np.empty(cout, np.float32)
    hip.d2h(dw, bufs[3])
    hip.d2h(db, bufs[4])
    for b in bufs:
        hip.free(b)
    ref_w, ref_b = osur.conv3x3_weight_grad(_dec(_enc(x, elem), elem), _dec(_enc(dz, elem), elem))
    for got, ref in ((dw, ref_w.transpose(0, 2, 1)), (db, ref_b)):
        assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)


@pytest.mark.parametrize("N,H,W", [(1, 1, 16), (1, 5, 48), (2, 7, 96), (9, 130, 64)])
@pytest.mark.parametrize("cin,cout,epi", [(64, 32, 0), (32, 32, 0), (64, 64, 0), (32, 64, 1), (64, 32, 2), (64, 64, 2)])
def test_conv_strips(hip, N, H, W, cin, cout, epi, elem="float16"):
    rng = np.random.default_rng(H + W + cin + cout)
    x, z = rng.normal(size=(N, H, W, cin)), rng.normal(size=(N, H, W, cout))
    w, b = rng.normal(0.0, 0.05, (9, cin, cout)).astype(np.float32), rng.normal(size=cout).astype(np.float32)
    ow, ob = hip.upload(w), hip.upload(b)
    wpk = hip.malloc(9 * cin * cout * 2)
    hip.check(hip.lib.lbm_sur_pack(_p(ow), cin, cout, cin, cout, _p(wpk), _p(None), CODE[elem], hip.stream), "pack")
    ox, oz = hip.upload(_enc(x, elem)), hip.upload(_enc(z, elem))
    out = np.empty((N, H, W, cout), np.float32 if epi == 1 else np.float16)
    oo = hip.malloc(out.nbytes)
    hip.check(hip.lib.lbm_sur_conv(_p(ox), cin, _p(wpk), _p(ob), _p(oz), _p(oo), _p(None), cout, epi, N, H, W,
                                   CODE[elem], hip.stream), "conv")
    hip.d2h(out, oo)
    for q in (ow, ob, wpk, ox, oz, oo):
        hip.free(q)
    wr = _dec(_enc(w, elem), elem)
    ref = osur.conv3x3(_dec(_enc(x, elem), elem), wr, b.astype(np.float64) if epi < 2 else 0.0)
    if epi == 0:
        ref = osur.silu(ref)
    elif epi == 2:
        ref = ref * osur.silu_grad(_dec(_enc(z, elem), elem))
    tol = 1e-6 if epi == 1 else 2 * UNIT[elem]
    assert np.linalg.norm(out - ref) <= tol * np.linalg.norm(ref)


@pytest.mark.parametrize("elem", ["float16", "bfloat16"])
def test_adam_net_equals_adam_and_pack(hip, elem):
    from pylbm_amd import runtime
    rng = np.random.default_rng(3)
    shapes = [(64, 32), (32, 64)]
    layers, kept = (runtime.LbmSurLayer * 2)(), []
    for i, (ci, co) in enumerate(shapes):
        k = 9 * ci * co
        host = [rng.normal(size=n).astype(np.float32) for n in (k, co, k + co, k + co, k, co)]
        host[3] = np.abs(host[3])
        a, b = [hip.upload(h) for h in host], [hip.upload(h) for h in host]
        pa, pb = [hip.malloc(k * 2) for _ in range(2)], [hip.malloc(k * 2) for _ in range(2)]
        layers[i] = runtime.LbmSurLayer(*a, *pa, ci, co)
        hip.check(hip.lib.lbm_sur_adam(*[_p(q) for q in b], ci, co, ci, co, 1e-2, 0.9, 0.99, 1e-3, 3, hip.stream), "adam")
        hip.check(hip.lib.lbm_sur_pack(_p(b[0]), ci, co, ci, co, _p(pb[0]), _p(pb[1]), CODE[elem], hip.stream), "pack")
        kept.append((host, a, b, pa, pb, k))
    hip.check(hip.lib.lbm_sur_adam_net(layers, 2, 1e-2, 0.9, 0.99, 1e-3, 3, CODE[elem], hip.stream), "adam_net")
    for host, a, b, pa, pb, k in kept:
        for p, q, n, t in [(a[i], b[i], host[i].size, np.float32) for i in range(4)] + \
                [(pa[i], pb[i], k, np.uint16) for i in range(2)]:
            u, v = np.empty(n, t), np.empty(n, t)
            hip.d2h(u, p)
            hip.d2h(v, q)
            assert np.array_equal(u, v)
        for p in a + b + pa + pb:
            hip.free(p)
