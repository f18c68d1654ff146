"""The plain FP64 analysis with observation errors down to 1e-15 of the spread's
variance, so that the condition numbers go through the node table's rows up to
the last (2^47; the matrix transform's fourth group of 16 nodes from 2^33 on) and
past it, for groups of few slabs (the solves in two rounds of nodes) and of
many (the matrix).

Bound: each solver, the oracle's eigensolve too, changes the matrix A by some
units of 2.2e-16 of its norm, and so its smallest eigenvalue, k - 1 exactly (the
mean's direction), by as many of the condition number; the square root halves
that.  4 x 2.2e-16 x kappa, with the trace's bound of kappa (at least the number
itself, at most k times), on top of the 1e-10 of well-conditioned problems."""
import dataclasses

import numpy as np
import pytest

from helpers import oracle_run, rel
from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


def _kappa(p):
    """Least and largest trace bound of the condition numbers, from the selection."""
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        t = []
        for ij in range(0, p.nij, 5):
            if p.mask[ij]:
                continue
            idx, w = s.selection(ij, 0)
            y = p.hx[:, idx].astype(np.float64)
            t.append(1.0 + float(((y * y).sum(0) * w / p.oerr[idx]).sum()) / (p.k - 1))
    return min(t), max(t)


@pytest.mark.parametrize("ns", [1, 12])
@pytest.mark.parametrize("k", [20, 50, 63])
@pytest.mark.parametrize("err", [1e-6, 1e-9, 1e-11, 1e-13, 1e-15])
def test_small_errors(err, k, ns):
    p = synth.random_problem(seed=900 + k, nx=20, ny=10, k=k, ns=ns, nobs=1200)
    p = dataclasses.replace(p, oerr=np.full(p.nobs, err, np.float32))
    lo, hi = _kappa(p)
    print("conditioning", err, k, ns, "log2 of kappa between", np.log2(lo / k), np.log2(hi), flush=True)
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        st, mn, sp = s.state_f64()
    ref = oracle_run(p)
    tol = 1e-10 + 4 * 2.2e-16 * hi
    e = dict(mean=rel(mn - p.mean, ref["mean"] - p.mean), sprd=rel(sp, ref["sprd"]),
             pert=rel(st - mn[None], ref["state"] - ref["mean"][None]))
    print(e, "tol", tol, flush=True)
    assert max(e.values()) <= min(tol, 0.5), (e, tol)
