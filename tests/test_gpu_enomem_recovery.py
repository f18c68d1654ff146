"""A set call or a run that runs out of device memory at any of its allocations
leaves a handle that refuses to run (LETKF_ESTATE) or runs to the right
analysis, and that can be set up again: the observations grow past the
handle's buffers, the localizer from one group to 26, under caps from what the
small analysis needs to what the large one does."""
import numpy as np
import pytest

from letkf_amd import abi, synth
from letkf_amd.solver import LetkfError, LetkfGpuSolver

pytestmark = pytest.mark.gpu


def _set(s, p):
    """Every input of p that can differ, each call on its own; the failures' codes."""
    s.prob = p
    bad = []

    def tried(f):
        try:
            f()
        except LetkfError as e:
            bad.append(e.code)

    def localizer():
        desc, keep = p.loc.to_c()
        s._chk(s.lib.letkf_gpu_set_localizer(s.h, desc))
        del keep

    tried(s._upload_obs)
    tried(localizer)
    return bad


def _run(s):
    try:
        s.run()
    except LetkfError as e:
        return e.code
    return s.state_f64()


@pytest.mark.parametrize("path,prec", [("plain", "fp64"), ("batched", "bf16x3")])
def test_caps_between_a_small_and_a_large_analysis(path, prec, monkeypatch):
    small = synth.random_problem(seed=11, nx=18, ny=9, k=12, ns=26, nobs=300)
    large = synth.random_problem(seed=12, nx=18, ny=9, k=12, ns=26, nobs=9000, radius=900e3,
                                 loc_cls="LOC_VGAUSS")
    large.state, large.mean, large.sprd = small.state, small.mean, small.sprd
    # one variable of 26 levels for both: the localizer's groups
    small.var_s, small.var_lev, small.inc_max, small.bounds = (large.var_s, large.var_lev, large.inc_max,
                                                               large.bounds)
    ref = {}
    for n, p in (("small", small), ("large", large)):
        with LetkfGpuSolver(p, precision=prec, path=path) as s:
            ref[n] = _run(s)
    seen = {"set": 0, "run": 0, "state": 0, "whole": 0, "back": 0}
    for cap in range(3 << 20, 60 << 20, 700 << 10):
        monkeypatch.setenv("LETKF_GPU_MEM_LIMIT", str(cap))
        try:
            s = LetkfGpuSolver(small, precision=prec, path=path)
        except LetkfError as e:
            assert e.code == abi.LETKF_ENOMEM
            continue
        with s:
            print("cap", cap >> 10, path, flush=True)
            got = _run(s)
            if isinstance(got, int):
                assert got == abi.LETKF_ENOMEM
                continue
            for name, p in (("large", large), ("small", small), ("large", large)):
                bad = _set(s, p)
                assert all(c == abi.LETKF_ENOMEM for c in bad)
                got = _run(s)
                seen["set"] += bool(bad)
                if isinstance(got, int):
                    # a failed set call: nothing to run on, unless the call failed before it
                    # let go of the old inputs
                    assert got in (abi.LETKF_ENOMEM, abi.LETKF_ESTATE)
                    seen["state" if got == abi.LETKF_ESTATE else "run"] += 1
                elif not bad:
                    for a, b in zip(got, ref[name]):
                        assert np.array_equal(a, b)
                    seen["whole" if name == "large" else "back"] += 1
    print(seen, flush=True)
    assert min(seen.values()) > 0
