"""Arrays of 8 MB and more that the runtime knows, handed to the setters and the
getters in the place of pageable ones: device tensors (a copy between two
device addresses) and a page-locked array.  The large-copy threads serve
memory of the host alone; everything the runtime knows goes its way.  The
analysis is the pageable call's bit for bit."""
import ctypes as C

import numpy as np
import pytest
import torch

from letkf_amd import abi, synth
from letkf_amd.solver import LetkfGpuSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["device", "locked"])
def test_arrays_the_runtime_knows(where):
    p = synth.random_problem(seed=91, nx=211, ny=103, k=51, ns=2, nobs=43001, radius=150e3)
    F, I = C.c_float, C.c_int32
    assert min(p.state.nbytes, p.hx.nbytes) >= 8 << 20

    def known(a):
        t = torch.from_numpy(np.ascontiguousarray(a.T))
        return t.cuda() if where == "device" else t.pin_memory()

    def at(t):
        return C.cast(t.data_ptr(), C.POINTER(F))

    with LetkfGpuSolver(p, precision="fp64", path="plain") as s:
        s.run()
        ref = [np.zeros(sh, np.float32, order="F") for sh in ((p.k, p.ns, p.nij), (p.ns, p.nij), (p.ns, p.nij))]
        s._chk(s.lib.letkf_gpu_get_state(s.h, *(abi.ptr(a, F) for a in ref)))
        ref_members = s.state_members()
        st, hx = known(p.state), known(p.hx)
        print("known", where, p.state.nbytes, p.hx.nbytes, flush=True)
        torch.cuda.synchronize()
        s._chk(s.lib.letkf_gpu_set_state(s.h, at(st), abi.ptr(p.mean, F), abi.ptr(p.sprd, F),
                                         abi.ptr(p.lat, F), abi.ptr(p.lon, F), abi.ptr(p.mask, I)))
        s._chk(s.lib.letkf_gpu_set_obs(
            s.h, p.nobs, abi.ptr(p.olat, F), abi.ptr(p.olon, F), abi.ptr(p.ozdim, F),
            abi.ptr(p.otime, F), abi.ptr(p.oval, F), abi.ptr(p.oerr, F), abi.ptr(p.obsid, I),
            abi.ptr(p.platid, I), at(hx), abi.ptr(p.hxmean, F)))
        s.run()
        got = [known(np.zeros_like(a)) for a in ref]
        torch.cuda.synchronize()
        s._chk(s.lib.letkf_gpu_get_state(s.h, *(at(t) for t in got)))
        torch.cuda.synchronize()
        for a, t in zip(ref, got):
            assert np.array_equal(t.cpu().numpy().T, a)
        got = [known(np.zeros_like(a)) for a in ref_members]
        torch.cuda.synchronize()
        s._chk(s.lib.letkf_gpu_get_state_members(s.h, *(at(t) for t in got)))
        torch.cuda.synchronize()
        for a, t in zip(ref_members, got):
            assert np.array_equal(t.cpu().numpy().T, a)
