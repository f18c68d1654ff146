"""The node tables that the build writes as constants (gen_ratnodes.cpp): value
for value what ratnodes.h computes, the stated errors row by row in extended
precision, and no library source that would compute them when it runs."""
import ctypes as C
import glob
import os
import re
import subprocess

import numpy as np
import pytest

from letkf_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))
NB, LD = 48, 128


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("gen"))
    text = open(build.generate(d)).read()
    body = re.search(r"kRatTab\[[^]]*\] = \{(.*?)\};", text, re.S).group(1)
    tab = np.array([float.fromhex(v) for v in body.replace("\n", "").split(",") if v])
    n = np.array(re.search(r"kRatN\[[^]]*\] = \{(.*?)\};", text, re.S).group(1).replace("\n", "").split(",")[:-1],
                 dtype=int)
    assert tab.size == 2 * NB * LD and n.size == 2 * NB
    return tab.reshape(2, NB, LD), n.reshape(2, NB)


def test_values(tables, tmp_path):
    tab, n = tables
    so = str(tmp_path / "librn.so")
    subprocess.run(["g++", "-O2", "-fPIC", "-shared", "-std=c++17",
                    os.path.join(HERE, "native", "ratnodes_host.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)
    lib.rn_nodes.argtypes = [C.c_double, C.c_int, C.POINTER(C.c_double), C.POINTER(C.c_double)]
    for b in range(1, NB):
        m = n[0, b]
        s, w = np.zeros(64), np.zeros(64)
        lib.rn_nodes(2.0 ** b, int(m), s.ctypes.data_as(C.POINTER(C.c_double)),
                     w.ctypes.data_as(C.POINTER(C.c_double)))
        # two compilers, each with its own library's last bit
        assert np.allclose(tab[0, b, :64], s, rtol=1e-14, atol=0) and np.allclose(tab[0, b, 64:], w, rtol=1e-14, atol=0)


def test_stated_errors(tables):
    tab, n = tables
    assert n[0, 1:].max() == 31 and n[1, 1:].max() == 62
    L = np.longdouble
    for b in range(1, NB):
        x = np.exp(np.log(L(2.0) ** b) * np.linspace(0, 1, 3001, dtype=L))
        for t in (0, 1):
            m = n[t, b]
            s, w = tab[t, b, :m].astype(L), tab[t, b, 64:64 + m].astype(L)
            err = float(np.abs((w[None] / (x[:, None] + s[None])).sum(1) * np.sqrt(x) - 1).max())
            if t == 0:
                assert err <= (1e-12 if b <= 26 else 1.8e-12 * 2.5 ** (b - 27)), (b, err)
            else:
                assert err <= (6e-16 if b <= 42 else 3e-14), (b, err)


def test_the_library_computes_none():
    for f in glob.glob(os.path.join(build.CSRC, "*.hip")) + glob.glob(os.path.join(build.CSRC, "*.h")):
        if os.path.basename(f) != "ratnodes.h":
            assert '#include "ratnodes.h"' not in open(f).read(), f
