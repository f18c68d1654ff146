"""The order of the padded observation columns follows the products that read
them: a handle whose tile choice changes between runs on the same observations
(the columns are put in the other order), and one that gets new observations
under either choice, give what handles made with that choice give, bit for
bit.  k + 1 of one row tile and over, odd and even numbers of tiles, the last
with 16-row tiles and the first without."""
import numpy as np
import pytest

from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


def _analyse(s):
    s.run()
    return s.state_f64()


def _same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("prec", ["bf16x4", "fp32"])
@pytest.mark.parametrize("k", [9, 15, 16, 33, 50, 64, 111, 112])
def test_tile_choice_between_runs(k, prec, monkeypatch):
    p = synth.random_problem(seed=300 + k, nx=24, ny=12, k=k, ns=1, nobs=1001)
    q = synth.random_problem(seed=301 + k, nx=24, ny=12, k=k, ns=1, nobs=703)
    ref = {}
    for tile in (0, 1):
        monkeypatch.setenv("LETKF_GPU_TILE", str(tile))
        for n, x in (("p", p), ("q", q)):
            with LetkfGpuSolver(x, precision=prec, path="batched") as s:
                ref[n, tile] = _analyse(s)
    with LetkfGpuSolver(p, precision=prec, path="batched") as s:
        for tile in (1, 0, 0, 1):
            print("order", k, prec, tile, flush=True)
            s.set_tuning(order=3, tile=tile)
            _same(_analyse(s), ref["p", tile])
        s.set_tuning(order=3, tile=0)
        s.cycle(q)                                  # new observations under the other choice
        _same(_analyse(s), ref["q", 0])
        s.set_tuning(order=3, tile=1)
        s.run_graph()
        s.run_graph()
        _same(s.state_f64(), ref["q", 1])
