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


@pytest.mark.parametrize("pad", [0, 8])
def test_captured_many_queries(torch_dev, pad):
    """The same for the many-query kernels' partials (64 queries: 15.7 MB at
    8,300 tokens, 17.3 MB at 8,192), a larger query count (a longer descriptor
    list) and, with padded rows, the operator's copies of them.  That the old
    buffers are still allocated is seen from the free memory before the graph
    runs again."""
    torch = torch_dev
    heads, dim, full, short, nq = 8, 128, 8300, 8192, 64
    g = torch.Generator(device="cuda").manual_seed(pad)
    k, v = (torch.randn(heads, full, dim, generator=g, device="cuda") for _ in range(2))
    q = torch.randn(2 * nq, heads, dim + pad, generator=g, device="cuda")
    m = L.adaptq_mha_create(heads, dim, 4, 4, full, 42, 0.0, 0)
    assert m, err()
    rows = {n: (k[:, :n].contiguous(), v[:, :n].contiguous()) for n in (full, short)}

    def fill(n):
        assert L.adaptq_mha_append_all_device(m, *map(_ptr, rows[n]), n, 0, None) == 0, err()
        torch.cuda.synchronize()

    def decode(out, n_queries, stream=None):
        row = 4 * (dim + pad)
        return L.adaptq_ggml_attn_f32_device(m, _ptr(q), dim, heads, n_queries, row, heads * row,
                                             _ptr(out), row, heads * row, stream) >= 0

    want, got, other = (torch.zeros_like(q) for _ in range(3))
    fill(full)
    assert decode(want, nq), err()
    torch.cuda.synchronize()
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        ok = decode(got, nq, C.c_void_p(s.cuda_stream))
    assert ok, err()
    for count in (nq, 2 * nq):
        L.adaptq_mha_reset(m)
        fill(short)
        before = torch.cuda.mem_get_info()[0]
        assert decode(other, count), err()
        torch.cuda.synchronize()
        # the new workspace alone takes over 16 MB, if no old one was freed for it
        if count == nq:
            assert before - torch.cuda.mem_get_info()[0] >= 16 << 20
        L.adaptq_mha_reset(m)
        fill(full)
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got[:nq], want[:nq]) and not got[nq:].any()
    del graph
    L.adaptq_mha_destroy(m)
