"""The search's short distance and Gaspari-Cohn weight (det_math.h: fewer
operations, with a flag that the float is the full form's) against the full
forms, on the CPU: where the flag is set the floats are the same, and it is
rarely not set.  The host's estimates of 1/sqrt and 1/x are at least as
coarse as the device's."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "search_fast_host.cpp")
HDR = os.path.join(HERE, "..", "umd-letkf_amd", "csrc", "det_math.h")
OUT = os.path.join(HERE, "native", "_build", "libsearchfast.so")


@pytest.fixture(scope="module")
def lib():
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    if not os.path.exists(OUT) or os.path.getmtime(OUT) < max(os.path.getmtime(SRC),
                                                              os.path.getmtime(HDR)):
        subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "-march=native", "-fPIC", "-shared", "-std=c++17",
                        "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", SRC, "-o", OUT],
                       check=True)
    return C.CDLL(OUT)


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def _count(fn, n, *arrays):
    wrong, unsure = C.c_long(), C.c_long()
    fn(C.c_long(n), *(_ptr(a) for a in arrays), C.byref(wrong), C.byref(unsure))
    return wrong.value, unsure.value / n


@pytest.mark.parametrize("top", [1e-8, 1e-4, 2.3e-3, 0.043 * 4])
def test_distance(lib, top):
    g = np.random.default_rng(1)
    n = 2_000_000
    c2 = np.concatenate([g.uniform(0.0, top, n // 2), top * 10.0 ** g.uniform(-12, 0, n // 2)])
    wrong, unsure = _count(lib.sfh_dist, n, c2)
    assert wrong == 0
    assert unsure < 1e-5
    assert _count(lib.sfh_dist, 1, np.zeros(1)) == (0, 1.0)      # no estimate: the full form


@pytest.mark.parametrize("L", [200e3 / 3.65, 82.2e3, 500e3, 720e3])
def test_weight(lib, L):
    g = np.random.default_rng(2)
    n = 4_000_000
    c = L / np.sqrt(0.3)
    z = np.concatenate([
        g.uniform(0.0, 2.1 * c, n // 2),
        c * g.uniform(1.8470, 1.8476, n // 4),                   # about the keep threshold
        c * (1.0 + g.uniform(-1e-6, 1e-6, n // 8)),              # the two polynomials' seam
        c * (2.0 + g.uniform(-1e-5, 1e-6, n // 8))]).astype(np.float32)
    Ls = np.full(n, L, np.float32)
    wrong, unsure = _count(lib.sfh_gc, n, z, Ls)
    assert wrong == 0
    assert unsure < 0.01
    z0 = np.zeros(1, np.float32)
    assert _count(lib.sfh_gc, 1, z0, Ls[:1])[0] == 0
