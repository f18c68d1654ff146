"""The large-ensemble transform with one row a lane at the edges of its row
lengths (72, 80, .. 104: just full and one over, where k > 104 is the 2D-block
kernels'), of the first wave's 64 rows, and of the blocks of 16 columns, with
lists shorter than k (many zero columns: reflectors left out) and long ones.
The plain FP64 path meets the oracle to 1e-10, the bar of that path."""
import numpy as np
import pytest

from helpers import oracle_run, rel
from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nobs", [25, 1200])
@pytest.mark.parametrize("k", [64, 65, 66, 72, 73, 79, 80, 81, 88, 89, 95, 96, 97, 100, 104, 105])
def test_row_lengths(k, nobs):
    p = synth.random_problem(seed=9000 + k, nx=18, ny=9, k=k, ns=3, nobs=nobs, rtps=0.3)
    orc = oracle_run(p)
    print("row transform k", k, "nobs", nobs, flush=True)
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        st, mn, sp = s.state_f64()
        hs = s.diag()["lg_selhash"]
    assert np.array_equal(hs.T, orc["lg_hash"])
    e = dict(mean=rel(mn, orc["mean"]), sprd=rel(sp, orc["sprd"]), state=rel(st, orc["state"]))
    assert max(e.values()) <= 1e-10, e
