"""Whether a caller's array is one page-locked allocation's (host_memory.h),
against the allocations byte by byte: arrays inside one, past its end, over
two with ordinary memory or nothing between them, and pageable ones, with the
device's addresses equal to the host's and elsewhere."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "host_memory_host.cpp")
OUT = os.path.join(HERE, "native", "_build", "libhost_memory.so")


@pytest.fixture(scope="module")
def hm():
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    subprocess.run(["g++", "-O2", "-fPIC", "-shared", "-std=c++17", SRC, "-o", OUT], check=True)
    lib = C.CDLL(OUT)
    P, Z = C.POINTER(C.c_void_p), C.POINTER(C.c_size_t)
    lib.hm_locked_span.restype = C.c_void_p
    lib.hm_locked_span.argtypes = [C.c_void_p, C.c_size_t, C.c_int, P, P, Z]
    return lib


@pytest.mark.parametrize("shift", [0, 1 << 20])
def test_locked_span(hm, shift):
    host = [4096, 3 * 4096, 4 * 4096]               # a gap after the first, none after the second
    size = [4096, 4096, 100]
    n = len(host)
    ha, da = (C.c_void_p * n)(*host), (C.c_void_p * n)(*(h + shift for h in host))
    sa = (C.c_size_t * n)(*size)
    for p in (4000, 4096, 4097, 8000, 8191, 8192, 12288, 16000, 16384, 16483, 16484):
        for m in (1, 2, 95, 100, 101, 192, 4095, 4096, 4097, 4196, 8192, 12288, 12389):
            inside = any(h <= p and p + m <= h + s for h, s in zip(host, size))
            got = hm.hm_locked_span(p, m, n, ha, da, sa)
            assert got == (p + shift if inside else None), (p, m)
    assert hm.hm_locked_span(4096, 0, n, ha, da, sa) is None
    assert hm.hm_locked_span(None, 4, n, ha, da, sa) is None
