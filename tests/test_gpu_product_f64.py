"""The FP64 products at the edges of their kernels: row blocks that are just
full (k + 1 a multiple of 16) or hold one row, few problems a chunk (four waves
share a problem's observations) and many (one wave each), tiles shared by four
waves (k >= 64), and lists of 1 observation to some hundreds (batches of 64, steps
of 4).  The plain FP64 path meets the oracle to 1e-10, the bar of that path."""
import numpy as np
import pytest

from helpers import oracle_run, rel
from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,nx,ny,nobs", [
    (15, 27, 13, 900), (16, 27, 13, 900), (47, 27, 13, 60), (63, 27, 13, 2000),
    (15, 97, 49, 900), (31, 97, 49, 9000), (48, 97, 49, 40), (63, 97, 49, 900),
    (64, 27, 13, 900), (79, 27, 13, 900), (80, 27, 13, 60), (96, 27, 13, 900),
    (111, 27, 13, 900), (127, 27, 13, 1500)])
def test_edges(k, nx, ny, nobs):
    p = synth.random_problem(seed=7000 + 8 * k + nx, nx=nx, ny=ny, k=k, ns=1, nobs=nobs, rtps=0.3)
    pts = np.arange(0, p.nij, 1 if nx < 50 else 29)
    orc = oracle_run(p, points=pts)
    print("product f64 k", k, "nij", p.nij, "nobs", nobs, flush=True)
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        st, mn, sp = s.state_f64()
        hs = s.diag()["lg_selhash"]
        print("problems", s.timing()["n_problems"], flush=True)
    assert np.array_equal(hs[pts].T, orc["lg_hash"])
    e = dict(mean=rel(mn[:, pts], orc["mean"]), sprd=rel(sp[:, pts], orc["sprd"]),
             state=rel(st[:, :, pts], orc["state"]))
    assert max(e.values()) <= 1e-10, e
