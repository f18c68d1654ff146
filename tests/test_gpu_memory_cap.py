"""LETKF_GPU_MEM_LIMIT bounds all that a handle holds, the blocks it keeps
between calls among it, and an analysis that fits the cap runs: the kept
blocks and the table of vertical weights make room for the lists and work
arrays.  Without the table the search evaluates the weights: the same lists
and analysis bit for bit."""
import numpy as np
import pytest
import torch

from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


def _analyse(s):
    s.run()
    return (*s.state_f64(), s.diag())


def _same(a, b):
    for x, y in zip(a[:3], b[:3]):
        assert np.array_equal(x, y)
    for n in a[3]:
        assert np.array_equal(a[3][n], b[3][n])


def test_weight_table_makes_room(monkeypatch):
    """120 000 observations on 50 levels: 30 MB of weights, 235 MB of lists, 33 MB
    of the rest and 15 MB of an upload's temporaries.  The cap holds all but the table."""
    p = synth.random_problem(seed=5, nx=18, ny=9, k=4, ns=50, nobs=120000, radius=900e3,
                             loc_cls="LOC_VGAUSS")
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        ref = _analyse(s)
        ref_sel = s.selection(40, 7)
    monkeypatch.setenv("LETKF_GPU_MEM_LIMIT", str(285 << 20))
    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        print("capped", flush=True)
        _same(_analyse(s), ref)
        for a, b in zip(s.selection(40, 7), ref_sel):
            assert np.array_equal(a, b)
        s.cycle(p)
        _same(_analyse(s), ref)
        s.run_graph()
        s.run_graph()
        _same((*s.state_f64(), s.diag()), ref)


def test_kept_blocks_count(monkeypatch):
    """About 90 MB of observations and 125 MB of their upload's temporaries, which
    are kept; then 130 MB of the run's arrays, for which they make room."""
    cap = 290 << 20
    p = synth.random_problem(seed=6, nx=100, ny=50, k=50, ns=10, nobs=200000, radius=60e3)
    g = np.random.default_rng(6)
    hx = np.asfortranarray(p.hx + p.hxmean[None])
    qc = (g.random(p.nobs) < 0.1).astype(np.int32)
    with LetkfGpuSolver(p, precision="fp64", path="plain", obs_members=(qc, hx)) as s:
        ref = _analyse(s)
    monkeypatch.setenv("LETKF_GPU_MEM_LIMIT", str(cap))
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    with LetkfGpuSolver(p, precision="fp64", path="plain", obs_members=(qc, hx)) as s:
        _same(_analyse(s), ref)
        held = free - torch.cuda.mem_get_info()[0]
        print("held", held >> 20, "of", cap >> 20, "MB", flush=True)
        assert held <= cap + (32 << 20)                # the driver's own rounding
