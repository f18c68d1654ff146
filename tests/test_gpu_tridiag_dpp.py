"""The DPP tridiagonalization at the edges of its kernels: every row length
(8 to 64), one and two rows a lane, one and two problems a wave, and carried
vectors that fill the spare rows exactly, do not fit them (k + NV > 32, k + NV
> 64) or are not carried at all (more than 8 slabs).  The FP64 path meets the
oracle to 1e-10 and the batched path's mean and spread to 1e-5, the bars of
those paths; the grid has an odd number of gridpoints."""
import numpy as np
import pytest

from helpers import oracle_run, rel
from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,ns", [(2, 1), (7, 8), (8, 1), (9, 2), (16, 4), (20, 1), (23, 8),
                                  (24, 8), (25, 8), (30, 1), (30, 2), (31, 1), (31, 9), (32, 1),
                                  (33, 8), (48, 3), (50, 8), (51, 1), (56, 8), (57, 4), (59, 4),
                                  (60, 4), (62, 1), (63, 1), (63, 8), (63, 10)])
def test_edges(k, ns):
    p = synth.random_problem(seed=400 + 16 * k + ns, nx=27, ny=13, k=k, ns=ns, nobs=1200, rtps=0.3)
    orc = oracle_run(p)
    for precision, path, tol in (("fp64", "plain", 1e-10), ("bf16x4", "batched", 1e-5)):
        print("tridiag dpp k", k, "ns", ns, precision, flush=True)
        with LetkfGpuSolver(p, precision=precision, path=path) as s:
            s.run()
            st, mn, sp = s.state_f64()
            hs = s.diag()["lg_selhash"]
        assert np.array_equal(hs.T, orc["lg_hash"])
        e = dict(mean=rel(mn, orc["mean"]), sprd=rel(sp, orc["sprd"]))
        if precision == "fp64":
            e["state"] = rel(st, orc["state"])
        print(e, flush=True)
        assert max(e.values()) <= tol, e


@pytest.mark.parametrize("rat", ["1", "0"])
@pytest.mark.parametrize("err", [0.05, 3e-3, 3e-4])
@pytest.mark.parametrize("k,ns", [(20, 1), (20, 12), (50, 1), (50, 12), (63, 2), (63, 12)])
def test_conditioning(k, ns, err, rat, monkeypatch):
    """The rational A^(-1/2) of the FP64 path with few and with many slabs a
    group, at condition numbers of the local problems up to about 8e6, which
    take more than one round of nodes (31) and more than one group of them
    (16), and the QL eigensolve it replaced (LETKF_GPU_RAT=0): both within
    1e-10 of the oracle."""
    monkeypatch.setenv("LETKF_GPU_RAT", rat)
    p = synth.random_problem(seed=1300 + k, nx=27, ny=13, k=k, ns=ns, nobs=1500, err=err, rtps=0.0)
    orc = oracle_run(p)
    print("conditioning k", k, "ns", ns, "err", err, "rat", rat, flush=True)
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        st, mn, sp = s.state_f64()
    e = dict(mean=rel(mn, orc["mean"]), sprd=rel(sp, orc["sprd"]), state=rel(st, orc["state"]),
             inc=rel(mn - p.mean, orc["mean"] - p.mean))
    print(e, flush=True)
    assert max(e.values()) <= 1e-10, e
