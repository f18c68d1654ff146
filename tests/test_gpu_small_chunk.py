"""Chunks whose list offsets and problem order one block makes, at the sizes
where it starts and ends (8192 and 16384 pairs, one over, ragged, two groups)
against the same analysis in gridpoint order (LETKF_GPU_BUCKET=0): the order of
the problems changes no bit, in eager runs and graph replays, and the
selection is the oracle's."""
import numpy as np
import pytest

from helpers import oracle_run
from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,loc", [(5, 3, "LOC_NOVRT"), (31, 33, "LOC_NOVRT"), (128, 64, "LOC_NOVRT"),
                                       (2731, 3, "LOC_NOVRT"), (128, 128, "LOC_NOVRT"),
                                       (565, 29, "LOC_NOVRT"), (64, 32, "LOC_OCEAN"), (91, 45, "LOC_OCEAN")])
def test_offsets_and_order(nx, ny, loc, monkeypatch):
    p = synth.random_problem(seed=500 + nx, nx=nx, ny=ny, k=12, ns=2, nobs=1500, loc_cls=loc)

    def run(bucket):
        monkeypatch.setenv("LETKF_GPU_BUCKET", bucket)
        with LetkfGpuSolver(p, precision="bf16x4", path="batched") as s:
            print("small chunk", nx, ny, loc, bucket, flush=True)
            s.run()
            out = [s.state_f64()]
            for _ in range(4):
                s.run_graph()
                out.append(s.state_f64())
            return out, s.diag()

    got, d = run("3")
    ref, _ = run("0")
    for o in got + ref[1:]:
        for a, b in zip(o, ref[0]):
            assert np.array_equal(a, b)
    pts = np.arange(0, p.nij, max(1, p.nij // 200))
    assert np.array_equal(d["lg_selhash"][pts].T, oracle_run(p, points=pts)["lg_hash"])
