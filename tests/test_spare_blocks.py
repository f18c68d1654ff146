"""The blocks a handle keeps between calls (spare_blocks.h): the best fit within
the bounds asked for, at most so many bytes and blocks with the oldest given
back first, one handle's blocks given back to a thread whose allocation
failed, nothing lost or given back twice with several threads."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "spare_blocks_host.cpp")
OUT = os.path.join(HERE, "native", "_build", "libspare_blocks.so")


@pytest.fixture(scope="module")
def sb():
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    subprocess.run(["g++", "-O2", "-fPIC", "-shared", "-std=c++17", "-pthread", SRC, "-o", OUT], check=True)
    lib = C.CDLL(OUT)
    H, P, Z = C.c_void_p, C.c_ssize_t, C.c_size_t
    lib.sb_new.restype, lib.sb_take.restype, lib.sb_bytes.restype, lib.sb_most.restype = H, P, Z, Z
    lib.sb_threads.restype = C.c_long
    lib.sb_keep.argtypes, lib.sb_take.argtypes = [H, P, Z], [H, Z, Z, C.POINTER(Z)]
    for f in ("sb_delete", "sb_bytes", "sb_release"):
        getattr(lib, f).argtypes = [H]
    return lib


def freed(sb):
    out = (C.c_ssize_t * 200)()
    return list(out[:sb.sb_freed(out, 200)])


def take(sb, h, least, most):
    size = C.c_size_t()
    p = sb.sb_take(h, least, most, C.byref(size))
    return (p, size.value) if p else None


def test_best_fit_and_bounds(sb):
    h = sb.sb_new(0)
    for p, size in ((1, 100), (2, 60), (3, 80), (4, 300)):
        sb.sb_keep(h, p, size)
    assert take(sb, h, 70, 140) == (3, 80)
    assert take(sb, h, 70, 140) == (1, 100)
    assert take(sb, h, 70, 140) is None                 # 60 too small, 300 too large
    assert sb.sb_bytes(h) == 360 and freed(sb) == []
    sb.sb_delete(h)
    assert sorted(freed(sb)) == [2, 4]


def test_bytes_and_count_bounded_oldest_first(sb):
    h, most, count = sb.sb_new(0), sb.sb_most(), sb.sb_count()
    sb.sb_keep(h, 1, most // 2)
    sb.sb_keep(h, 2, most // 2)
    assert freed(sb) == []
    sb.sb_keep(h, 3, 1)                                 # the oldest makes room
    assert freed(sb) == [1] and sb.sb_bytes(h) == most // 2 + 1
    sb.sb_keep(h, 4, most + 1)                          # larger than all that is kept
    assert freed(sb) == [4]
    sb.sb_keep(h, 5, most)
    assert freed(sb) == [2, 3] and sb.sb_bytes(h) == most
    sb.sb_release(h)
    assert freed(sb) == [5] and sb.sb_bytes(h) == 0
    for i in range(count + 3):
        sb.sb_keep(h, 10 + i, 8)
    assert freed(sb) == [10, 11, 12] and sb.sb_bytes(h) == 8 * count
    sb.sb_delete(h)
    assert len(freed(sb)) == count


def test_other_handles_give_back(sb):
    a, b, c = sb.sb_new(0), sb.sb_new(0), sb.sb_new(1)
    for i, h in enumerate((a, b, c)):
        sb.sb_keep(h, 20 + i, 50)
    assert sb.sb_release_device(0) == 1
    assert sorted(freed(sb)) == [20, 21]
    assert (sb.sb_bytes(a), sb.sb_bytes(b), sb.sb_bytes(c)) == (0, 0, 50)
    assert sb.sb_release_device(0) == 0
    sb.sb_delete(b)
    sb.sb_keep(a, 30, 5)
    assert sb.sb_release_device(0) == 1 and freed(sb) == [30]
    sb.sb_delete(a)
    sb.sb_delete(c)
    assert freed(sb) == [22]


def test_threads(sb):
    assert sb.sb_threads(4, 20000) == 0
