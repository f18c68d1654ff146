"""Results written by the kernels into page-locked host memory against the
copies to pageable memory, bit for bit: arrays on 16 bytes and 4 or 8 bytes
past them, odd lengths (tails of the 16-byte stores), arrays left out, one
array page-locked and one not (the copies serve the whole call), nothing
written past an array's end; and the diagnostics of several groups in either
way (small grids by a kernel, larger ones by copies)."""
import ctypes as C

import numpy as np
import pytest
import torch

from letkf_amd import abi, synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


def _fetch(s, f64, pinned, shift, skip=()):
    """state, mean, spread through the C ABI into arrays `shift` values into
    their memory, with a guard value after them."""
    p = s.prob
    dt = torch.float64 if f64 else torch.float32
    ct = C.c_double if f64 else C.c_float
    out, ptrs = [], []
    for i, n in enumerate((p.k * p.ns * p.nij, p.ns * p.nij, p.ns * p.nij)):
        t = torch.full((n + shift + 5,), -77.0, dtype=dt, pin_memory=bool(pinned[i]))
        a = t.numpy()[shift:]
        out.append(a)
        ptrs.append(None if i in skip else abi.ptr(a, ct))
    get = s.lib.letkf_gpu_get_state_f64 if f64 else s.lib.letkf_gpu_get_state
    assert get(s.h, *ptrs) == 0
    return out


@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("nx,ny,k,ns", [(5, 3, 3, 1), (18, 9, 21, 3), (97, 49, 50, 2)])
def test_state_to_host(nx, ny, k, ns, f64):
    p = synth.random_problem(seed=61 + nx, nx=nx, ny=ny, k=k, ns=ns, nobs=300, rtps=0.4)
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        ref = _fetch(s, f64, (0, 0, 0), 0)
        for pinned, shift, skip in (((1, 1, 1), 0, ()), ((1, 1, 1), 1, ()), ((1, 1, 1), 3, (1,)),
                                    ((1, 1, 1), 2, (0, 2)), ((1, 0, 1), 1, ()), ((1, 1, 1), 0, (0, 1, 2))):
            print("to host", nx, ny, k, ns, f64, pinned, shift, skip, flush=True)
            got = _fetch(s, f64, pinned, shift, skip)
            for i, n in enumerate((p.k * p.ns * p.nij, p.ns * p.nij, p.ns * p.nij)):
                if i in skip:
                    assert np.all(got[i] == -77.0)
                else:
                    assert np.array_equal(got[i][:n], ref[i][:n]) and np.all(got[i][n:] == -77.0)


def test_diagnostics_both_ways():
    """26 groups: 18 x 9 gridpoints go by the kernel, 108 x 54 by copies; a
    gridpoint's fields are compared with its selection."""
    for nx, ny in ((18, 9), (108, 54)):
        p = synth.random_problem(seed=77, nx=nx, ny=ny, k=10, ns=26, nobs=2500, loc_cls="LOC_VGAUSS")
        with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
            s.run()
            d = s.diag()
            again = s.diag()
            for n in d:
                assert np.array_equal(d[n], again[n])
            G = s.maxgroups()
            assert d["lg_obscount"].shape == (p.nij, G)
            for ij in range(3, p.nij, p.nij // 7):
                for g in (0, G // 2, G - 1):
                    idx, w = s.selection(ij, g)
                    print("diag", nx, ij, g, len(idx), flush=True)
                    assert d["lg_obscount"][ij, g] == len(idx)
                    assert abs(d["lg_obsloc"][ij, g] - w.astype(np.float64).sum()) <= 1e-5 * max(1.0, len(idx))
