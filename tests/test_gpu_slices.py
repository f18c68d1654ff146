"""letkf_gpu_get_state into pageable arrays of several slices (16M values each,
the last one ragged) and, for the mean, of less than the large copy's 8 MB: the
FP64 analysis rounded to single precision, bit for bit, with nothing written
past the arrays' ends; fields left out."""
import ctypes as C

import numpy as np
import pytest

from letkf_amd import abi, synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


def test_slices():
    p = synth.random_problem(seed=31, nx=433, ny=211, k=63, ns=3, nobs=400, radius=300e3)
    n = (p.k * p.ns * p.nij, p.ns * p.nij, p.ns * p.nij)
    assert n[0] > 1 << 24 and n[0] % (1 << 24) and 4 * n[1] < 8 << 20
    F = C.c_float
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        ref = [a.ravel(order="F").astype(np.float32) for a in s.state_f64()]
        for skip in ((), (0,), (1, 2)):
            print("slices", skip, flush=True)
            out = [np.full(m + 3, -77.0, np.float32) for m in n]
            s._chk(s.lib.letkf_gpu_get_state(s.h, *(None if i in skip else abi.ptr(a, F)
                                                    for i, a in enumerate(out))))
            for i, (a, r) in enumerate(zip(out, ref)):
                if i in skip:
                    assert np.all(a == -77.0)
                else:
                    assert np.array_equal(a[:-3], r) and np.all(a[-3:] == -77.0)
