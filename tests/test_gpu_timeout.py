"""Who reports a sync-free wait that ran out of time: the flag that such a wait
leaves for the host is set from the host (tests/cpp/trsv_flag.cpp, built by
__graft_entry__.build())."""
import ctypes
import os

import pytest

import linearalgebra_amd as la
from helpers import ROOT

pytestmark = pytest.mark.gpu


def test_transposed_apply_reports_a_timeout(dev):
    """A wait of the transposed ILU apply that ran out of time (its flag set
    from the host) is that call's error, and the next call is good again."""
    import torch
    flag = ctypes.CDLL(os.path.join(ROOT, "tests", "cpp", "libtrsv_flag.so"))
    flag.flag_transposed_timeout.argtypes = [ctypes.c_void_p]
    P = la.Preconditioner(la.iluk(la.gen.poisson2d(40), 0), "ilu")
    r = torch.tensor(la.gen.uniform(1600, 31), device=dev)
    z, ref = torch.zeros_like(r), torch.zeros_like(r)
    P.apply_transpose(r, ref)
    assert flag.flag_transposed_timeout(P.h) == 1
    with pytest.raises(la.LaError) as e:
        P.apply_transpose(r, z)
    assert e.value.code == 7
    P.apply_transpose(r, z)
    P.apply(r, torch.zeros_like(r))
    assert torch.equal(z, ref)


def test_transposed_apply_captures(dev):
    """The transposed apply, its plans built, can be recorded into a graph,
    where nothing can be waited for."""
    import torch
    P = la.Preconditioner(la.iluk(la.gen.poisson2d(40), 0), "ilu")
    r = torch.tensor(la.gen.uniform(1600, 32), device=dev)
    z, ref = torch.zeros_like(r), torch.zeros_like(r)
    P.apply_transpose(r, ref)
    torch.cuda.synchronize()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    P.set_stream(s)
    with torch.cuda.graph(g, stream=s):
        P.apply_transpose(r, z)
    for k in range(4):
        r.copy_(torch.tensor(la.gen.uniform(1600, 33 + k), device=dev))
        z.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        P.apply_transpose(r, ref)
        torch.cuda.synchronize()
        assert torch.equal(z, ref), k
