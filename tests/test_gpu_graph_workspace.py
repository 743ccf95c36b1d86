"""A decode captured into a graph keeps its workspace while other calls on the
same plan or MHA need a larger one: split counts are not monotone in the ring's
length, so shorter rings can.  Replays after that equal the eager decode of the
same rings bit for bit (same kernels, same split count, fixed merge order)."""
import ctypes as C

import pytest

from adaptq_amd import _lib
from gpu_head import err

pytestmark = pytest.mark.gpu
L = _lib.lib


def _ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("heads,dim,full,short", [(8, 128, 8704, 8192), (48, 128, 8192, 2560)])
@pytest.mark.parametrize("whole_mha", [False, True])
def test_captured_workspace(torch_dev, heads, dim, full, short, whole_mha):
    torch = torch_dev
    g = torch.Generator(device="cuda").manual_seed(heads)
    k, v = (torch.randn(heads, full, dim, generator=g, device="cuda") for _ in range(2))
    q = torch.randn(heads, dim, generator=g, device="cuda")
    m = L.adaptq_mha_create(heads, dim, 4, 4, full, 42, 0.0, 0)
    assert m, err()
    ctx = [L.adaptq_mha_head(m, h) for h in range(heads)]
    p = L.adaptq_plan_create((C.c_void_p * heads)(*ctx), heads)
    assert p, err()

    def append(lo, hi):
        ks, vs = k[:, lo:hi].contiguous(), v[:, lo:hi].contiguous()
        assert L.adaptq_plan_append_device(p, _ptr(ks), _ptr(vs), hi - lo, lo, None) == 0, err()
        torch.cuda.synchronize()

    def decode(out, stream=None):
        if whole_mha:
            return L.adaptq_mha_compute_all_device(m, _ptr(q), _ptr(out), stream) >= 0
        return L.adaptq_plan_compute_device(p, _ptr(q), _ptr(out), stream) == 0

    want, got, other = (torch.empty_like(q) for _ in range(3))
    append(0, full)
    assert decode(want), err()
    torch.cuda.synchronize()
    need = L.adaptq_plan_workspace_bytes(p)
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        ok = decode(got, C.c_void_p(s.cuda_stream))
    assert ok, err()
    for _ in range(2):
        L.adaptq_mha_reset(m)
        append(0, short)
        assert L.adaptq_plan_workspace_bytes(p) > need  # what the test is about
        assert decode(other), err()
        append(short, full)
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    del graph
    L.adaptq_plan_destroy(p)
    L.adaptq_mha_destroy(m)
