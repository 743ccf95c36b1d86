"""Decode plans whose rings differ in length: the split count is chosen from
the sum of the lengths, splits past a short ring's end are empty, and a plan
captured into a graph without a workspace runs unsplit.  Against the oracle,
within 1e-4 norm-wise as every output test; split and unsplit decodes of the
same rings merge their softmax differently by rounding only (1e-5 here)."""
import ctypes as C

import numpy as np
import pytest

from adaptq_amd import _lib
from gpu_head import err, rel_err

pytestmark = pytest.mark.gpu
L = _lib.lib


def _plan(handles):
    p = L.adaptq_plan_create((C.c_void_p * len(handles))(*handles), len(handles))
    assert p, err()
    return p


def _ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("dim,kb,vb,lens", [
    (96, 3, 3, [1, 64, 65, 511, 512, 513, 2048, 6500, 0, 4097]),
    (128, 4, 2, [8192] + [100] * 40), (64, 4, 4, [5000, 1, 0, 4999, 2049] * 8),
    (200, 4, 2, [3000] + [17] * 70), (64, 16, 16, [3000, 10, 700]),
    (128, 2, 3, [0, 0, 700]), (64, 3, 2, [2047, 5, 64] * 9),
])
def test_uneven_rings(oracle, torch_dev, dim, kb, vb, lens):
    torch = torch_dev
    rng = np.random.default_rng(dim + len(lens))
    cap = max(lens)
    hs = [L.adaptq_create(dim, kb, vb, cap, 100 + i, 0.0, 0) for i in range(len(lens))]
    assert all(hs), err()
    rows = {}
    check = set(range(min(10, len(lens)))) | {len(lens) - 1}
    for i, n in enumerate(lens):
        if n:
            k = rng.standard_normal((1, n, dim)).astype(np.float32)
            v = rng.standard_normal((1, n, dim)).astype(np.float32)
            kd, vd, p1 = torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), _plan([hs[i]])
            assert L.adaptq_plan_append_device(p1, _ptr(kd), _ptr(vd), n, 0, None) == 0, err()
            torch.cuda.synchronize()
            L.adaptq_plan_destroy(p1)
            if i in check:
                rows[i] = (k[0], v[0])
    q = rng.standard_normal((len(lens), dim)).astype(np.float32)
    qd = torch.from_numpy(q).cuda()
    outs = torch.empty_like(qd)
    p = _plan(hs)
    # captured with no workspace in hand (a side stream), then eager
    s = torch.cuda.Stream()
    graph, cap_out = torch.cuda.CUDAGraph(), torch.empty_like(qd)
    torch.cuda.synchronize()
    need = L.adaptq_plan_workspace_bytes(p)
    lut = dim <= 256
    with torch.cuda.graph(graph, stream=s):
        rc = L.adaptq_plan_compute_device(p, _ptr(qd), _ptr(cap_out), C.c_void_p(s.cuda_stream))
    assert rc == 0 or not lut, err()
    assert L.adaptq_plan_compute_device(p, _ptr(qd), _ptr(outs), None) == 0, err()
    torch.cuda.synchronize()
    y = outs.cpu().numpy()
    for i in check:
        if lens[i] == 0:
            assert not y[i].any()
            continue
        o = oracle.head(dim, kb, vb, cap, 100 + i)
        for t in range(lens[i]):
            o.append(rows[i][0][t], rows[i][1][t], t)
        assert rel_err(y[i], o.compute(q[i])[0]) <= 1e-4, (i, lens[i])
    for _ in range(3):
        cap_out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        z = cap_out.cpu().numpy()
        assert np.abs(z - y).max() <= 1e-5 * np.abs(y).max(), need
    L.adaptq_plan_destroy(p)
    for h in hs:
        L.adaptq_destroy(h)
