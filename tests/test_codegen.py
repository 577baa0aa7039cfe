"""Generated HIP source: pair-parity factoring is detected for the MRT bases and
the printed transforms are exact (checked by evaluating the printed C sums in
Python on random populations)."""
import re

import numpy as np
import pytest

from pylbm_amd import cases
from pylbm_amd.generator.hip import _pairs, _row_parities, generate_source
from pylbm_amd.scheme import Scheme


@pytest.mark.parametrize("make", [lambda: cases.lid_cavity_d2q9(8), lambda: cases.taylor_green_d3q19(4),
                                  lambda: cases.d2q5q9_vectorial(8), lambda: cases.d1q3_advection(8)])
def test_parity_detected(make):
    spec = Scheme(make()).kernel_spec()
    ksym = _pairs(spec)
    assert ksym is not None
    assert _row_parities(spec.M, ksym) is not None
    assert "pair-factored=True" in generate_source(spec)


def _eval_block(src, start, end, env):
    body = src[src.index(start):]
    body = body[:body.index(end)]
    for line in body.splitlines():
        line = line.strip()
        mm = re.match(r"(?:const C |C )?(\w+) = (.*);$", line)
        if not mm:
            continue
        expr = re.sub(r"C\(([-0-9.e+]+)\)", r"(\1)", mm.group(2))
        env[mm.group(1)] = eval(expr, {}, env)
    return env


def test_printed_transforms_are_exact():
    spec = Scheme(cases.taylor_green_d3q19(4)).kernel_spec()
    src = generate_source(spec)
    M = np.array([[float(c) for c in r] for r in spec.M])
    iM = np.array([[float(c) for c in r] for r in spec.invM])
    rng = np.random.default_rng(1)
    f = rng.random(spec.ns)
    env = {"f%d" % k: f[k] for k in range(spec.ns)}
    kern = src[src.index("fused_step(const S*"):]
    env = _eval_block(kern, "const C p0", "const C q_", env)
    m = np.array([env["m%d" % i] for i in range(spec.ns)])
    assert np.allclose(m, M @ f, rtol=1e-14, atol=1e-14)
    m2 = rng.random(spec.ns)
    env2 = {"m%d" % i: m2[i] for i in range(spec.ns)}
    start = kern.index("const C r0") if "const C r0" in kern else kern.index("const C E")
    env2 = _eval_block(kern[start:], kern[start:start + 10], "G0[j] = Codec<S>::encode(", env2)
    g = np.array([env2["g%d" % k] for k in range(spec.ns)])
    assert np.allclose(g, iM @ m2, rtol=1e-13, atol=1e-14)


def test_fused_step_addresses_stores_by_element_index():
    """The step's stores take the index type of the launch: 32-bit byte offsets would wrap
    in a layout whose strides span 4 GiB with fewer than 2^31 elements."""
    src = generate_source(Scheme(cases.taylor_green_d3q19(4)).kernel_spec())
    kern = src[src.index("fused_step(const S*"):]
    kern = kern[:kern.index("\n}\n")]
    assert kern.count("fn + ((I)a.dst_off[") == 19
    assert "buffer_store" not in kern and "uint32_t)(cell" not in kern


def test_step_without_a_table_keeps_its_registers(tmp_path):
    """The loads of table entries stay out of the kernels that boxes without a table run: the
    D3Q6 FP64 step fits the 64 registers of 8 waves per SIMD (compiled here, not run)."""
    import os
    import subprocess
    from pylbm_amd import demos
    from pylbm_amd.generator.build import CSRC, HIPCC, HIPCC_FLAGS, INCLUDE
    src = tmp_path / "d3q6.hip"
    src.write_text(generate_source(Scheme(demos.advection_3d(1 / 8)[0]).kernel_spec()))
    flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    out = subprocess.run([HIPCC] + flags + ["-I" + INCLUDE, "-I" + CSRC, "--cuda-device-only", "-c", str(src), "-o",
                                            os.devnull, "-Rpass-analysis=kernel-resource-usage"],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, check=True).stdout
    vgprs = {}
    for line in out.splitlines():
        name = re.search(r"Function Name: (\S+)", line)
        if name:
            kernel = name.group(1)
        count = re.search(r"    VGPRs: (\d+)", line)
        if count:
            vgprs[kernel] = int(count.group(1))
    steps = {k: v for k, v in vgprs.items() if "fused_stepId" in k}   # FP64
    assert len(steps) >= 6 and min(steps.values()) <= 64
    wrap = [v for k, v in steps.items() if "fused_stepIdLb1E" in k]   # periodic fold
    assert sum(v <= 64 for v in wrap) >= len(wrap) // 2, steps


def test_rule_of_the_cached_stores(tmp_path):
    """The rule counts what a step stores, not the padding of the rows: 64^3 FP16 (19 MiB in
    rows padded to three times that) bypasses the caches, 128^3 FP32 (304 MiB) does not."""
    import ctypes
    import os
    import subprocess
    from pylbm_amd.generator.build import INCLUDE
    from pylbm_amd.runtime import LBM_F16D, LBM_F32, LBM_F64
    from pylbm_amd.storage import make_layout
    src = generate_source(Scheme(cases.taylor_green_d3q19(4)).kernel_spec())
    fn = src[src.index("static int stream_stores("):]
    fn = fn[:fn.index("\n}\n") + 3].replace("static int", 'extern "C" int', 1)
    cpp, so = tmp_path / "rule.cpp", str(tmp_path / "rule.so")
    cpp.write_text('#include "pylbm_hip.h"\nstatic int storage_elem_size(int s) { return s == %d ? 2 : s == %d ? 4 : 8; }\n'
                   % (LBM_F16D, LBM_F32) + fn)
    subprocess.run(["g++", "-shared", "-fPIC", "-I" + INCLUDE, str(cpp), "-o", so], check=True)
    rule = ctypes.CDLL(os.path.abspath(so)).stream_stores
    rule.argtypes = [ctypes.c_void_p, ctypes.c_int64]
    for n, storage, most, past in ((64, LBM_F16D, 176, 1), (72, LBM_F16D, 176, 0), (128, LBM_F16D, 176, 0),
                                   (160, LBM_F16D, 176, 1), (48, LBM_F32, 306, 1), (56, LBM_F32, 306, 0),
                                   (128, LBM_F32, 306, 0), (136, LBM_F32, 306, 1), (96, LBM_F64, 306, 0),
                                   (96, LBM_F64, 256, 1), (120, LBM_F32, 256, 0), (1024, LBM_F64, 306, 1)):
        for interleaved in (False, True):
            L = make_layout(19, (n + 2,) * 3, (1, 1, 1), storage, interleaved)
            assert rule(ctypes.byref(L), most) == past, (n, storage, most)
