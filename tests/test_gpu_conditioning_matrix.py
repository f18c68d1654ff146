"""test_gpu_conditioning's analyses for 64 <= k <= 127, where every group takes
the transform matrix: each register layout of its reduction and back-transform
at its smallest and largest k (LETKF_GPU_MATBLK=0: the column halves), with the
bound that is derived there."""
import dataclasses

import numpy as np
import pytest

from helpers import oracle_run, rel
from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver
from test_gpu_conditioning import _kappa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("err", [1e-6, 1e-9, 1e-11, 1e-13])
@pytest.mark.parametrize("k,matblk", [(64, 1), (72, 1), (73, 1), (88, 1), (100, 1), (104, 1),
                                      (105, 1), (112, 1), (113, 1), (127, 1),
                                      (64, 0), (81, 0), (112, 0), (127, 0)])
def test_small_errors(k, matblk, err, monkeypatch):
    monkeypatch.setenv("LETKF_GPU_MATBLK", str(matblk))
    p = synth.random_problem(seed=700 + k, nx=12, ny=8, k=k, ns=3, nobs=700)
    p = dataclasses.replace(p, oerr=np.full(p.nobs, err, np.float32))
    lo, hi = _kappa(p)
    print("conditioning", err, k, matblk, "log2 of kappa between", np.log2(lo / k), np.log2(hi),
          flush=True)
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        st, mn, sp = s.state_f64()
    ref = oracle_run(p)
    tol = 1e-10 + 4 * 2.2e-16 * hi
    e = dict(mean=rel(mn - p.mean, ref["mean"] - p.mean), sprd=rel(sp, ref["sprd"]),
             pert=rel(st - mn[None], ref["state"] - ref["mean"][None]))
    print(e, "tol", tol, flush=True)
    assert max(e.values()) <= min(tol, 0.5), (e, tol)
