"""The mixed products over every number of row tiles: the column entries of a
lane are read as one run (1 to 7 values a lane in the 16-row tiles, 1 to 4 in
the 32-row blocks), so k + 1 just full, one row over and in between, with lists
from one observation to some hundreds (steps of 32, list entries in groups of
8).  Errors against the FP64 path on the same selection: an entry of the
product is a sum of m terms, each rounded to 2^-24 (FP32), 2^-17 (split BF16)
or 2^-8 (BF16) of the operands; with observation errors near the spread the
condition number of the problems is a few hundred, which with sums that grow
like sqrt(m) stays below 1e-5, 1e-4 and 3e-2 of the largest perturbation."""
import numpy as np
import pytest

from helpers import rel
from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu

TOL = {"fp32": 1e-5, "bf16x4": 1e-5, "bf16x3": 1e-4, "bf16": 3e-2}


@pytest.mark.parametrize("k,nobs", [(10, 40), (15, 900), (16, 900), (31, 900), (32, 900), (47, 900),
                                    (48, 40), (50, 900), (63, 900), (64, 900), (79, 900), (80, 900),
                                    (95, 900), (96, 900), (111, 900), (112, 900), (127, 900)])
def test_row_tiles(k, nobs):
    p = synth.random_problem(seed=8100 + k, nx=27, ny=13, k=k, ns=1, nobs=nobs, rtps=0.3)

    def run(**kw):
        with LetkfGpuSolver(p, **kw) as s:
            s.run()
            st, mn, sp = s.state_f64()
            return st, mn, sp, s.diag()["lg_selhash"]

    st0, mn0, sp0, h0 = run(precision="fp64", path="plain")
    for prec, tol in TOL.items():
        print("columns", prec, "k", k, "nobs", nobs, flush=True)
        st, mn, sp, h = run(precision=prec, path="batched")
        assert np.array_equal(h, h0)
        e = dict(mean=rel(mn, mn0), sprd=rel(sp, sp0), pert=rel(st - mn[None], st0 - mn0[None]))
        assert max(e.values()) <= tol, (prec, e)
