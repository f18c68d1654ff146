"""Members and observations large enough for the threads of the bulk copy (8 MB
and more; the last piece ragged), up and down, through the tiled layout
kernels (gridpoints past the last tile of 64, observations past the last 32):
bit for bit the arithmetic of the reference's order in numpy, from pageable
and from page-locked arrays, on a second call that takes the kept blocks, and
through the no-allocation fetch."""
import numpy as np
import pytest
import torch

from letkf_amd import synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,k,ns,nobs", [(211, 103, 51, 2, 43001), (300, 175, 10, 4, 33), (129, 65, 127, 3, 16411)])
def test_members_and_observations(nx, ny, k, ns, nobs):
    p = synth.random_problem(seed=400 + k, nx=nx, ny=ny, k=k, ns=ns, nobs=nobs, radius=200e3)
    rng = np.random.default_rng(k)
    mem = np.asfortranarray(rng.normal(size=(p.nij, ns, k)).astype(np.float32) + 3.0)
    hx = np.asfortranarray(rng.normal(size=(k, nobs)).astype(np.float32) + 3.0)
    qc = (rng.random(nobs) < 0.2).astype(np.int32)

    def analyse(s):
        s.run()
        return s.state_members(), s.state_members_noalloc()

    with LetkfGpuSolver(p, precision="fp64", path="plain", members=mem, obs_members=(qc, hx)) as s:
        print("bulk", mem.nbytes, hx.nbytes, flush=True)
        first, noalloc = analyse(s)
        for a, b in zip(first, noalloc):
            assert np.array_equal(a, b)
        s.cycle(p, members=mem, obs_members=(qc, hx))          # kept blocks
        for a, b in zip(analyse(s)[0], first):
            assert np.array_equal(a, b)
        tm = torch.empty((k, ns, p.nij), dtype=torch.float32, pin_memory=True)
        tm.numpy().T[...] = mem
        th = torch.empty((nobs, k), dtype=torch.float32, pin_memory=True)
        th.numpy().T[...] = hx
        s.cycle(p, members=tm.numpy().T, obs_members=(qc, th.numpy().T))
        for a, b in zip(analyse(s)[0], first):
            assert np.array_equal(a, b)

    # the same analysis from the separate fields, in the reference's FP32 order
    def split(x, axis):
        x = np.moveaxis(x, axis, 0)
        mu = np.zeros(x.shape[1:], np.float32)
        for m in range(k):
            mu = mu + x[m]
        mu = mu / np.float32(k)
        d = x - mu
        dot = np.zeros_like(mu)
        for m in range(k):
            dot = dot + d[m] * d[m]
        return mu, d, np.sqrt(dot / np.float32(k - 1))

    mu, d, sd = split(mem, 2)
    hmu, hd, _ = split(hx, 0)
    on = qc <= 0
    import dataclasses
    q = dataclasses.replace(
        p, state=np.asfortranarray(d.transpose(0, 2, 1)), mean=np.asfortranarray(mu.T),
        sprd=np.asfortranarray(sd.T), hx=np.asfortranarray(hd[:, on]), hxmean=np.ascontiguousarray(hmu[on]),
        **{n: np.ascontiguousarray(getattr(p, n)[on])
           for n in ("olat", "olon", "ozdim", "otime", "oval", "oerr", "obsid", "platid")})
    with LetkfGpuSolver(q, precision="fp64", path="plain") as s:
        other, _ = analyse(s)
    for a, b in zip(other, first):
        assert np.array_equal(a, b)
