"""The many-query kernel at the edges of its tiles (16 tokens, 16 queries a
wave, 1, 2 or 4 query groups a block, slices of a step, splits over tokens)
and of the rule that takes it (7 queries: the LUT kernel), against the oracle:
within 1e-4 norm-wise, as every output test; the logits repeat the reference's
own fp32 steps, so plain N(0,1) rings stay far below."""
import ctypes as C

import numpy as np
import pytest

import mq_rule
from adaptq_amd import _lib
from golden import inputs as I
from gpu_head import err, rel_err

pytestmark = pytest.mark.gpu
L = _lib.lib


@pytest.mark.parametrize("dim,kb,vb", [(128, 4, 4), (128, 3, 3), (100, 2, 2), (64, 4, 3),
                                       (48, 3, 2), (64, 2, 4)])
@pytest.mark.parametrize("nq", [7, 8, 16, 17, 32, 33, 49, 64, 65])
def test_tile_edges(oracle, torch_dev, dim, kb, vb, nq):
    """As many heads as the kernel takes the call at (from 8 queries on); rings
    of whole tiles, one token more or less, a whole and a part step or split, and
    a wrapped one."""
    torch = torch_dev
    rng = np.random.default_rng(dim + 10 * kb + nq)
    sizes, cap, seed = (1023, 1024, 1025, 1037, 1281, 1500), 1300, 11 * dim + nq
    P = 64 if dim <= 64 else 128
    H = mq_rule.heads_for(nq, sizes[0], P) if nq >= 8 else 96
    assert all(mq_rule.takes(H, nq, min(n, cap), P) == (nq >= 8) for n in sizes)
    m = L.adaptq_mha_create(H, dim, kb, vb, cap, seed, 0.0, 0)
    assert m, err()
    check = (0, H // 2, H - 1)
    refs = {h: oracle.head(dim, kb, vb, cap, I.mha_seed(seed, h)) for h in check}
    qd = torch.from_numpy((rng.standard_normal((nq, H, dim)) * 2).astype(np.float32)).cuda()
    qs, od, row = qd.cpu().numpy(), torch.empty_like(qd), 4 * dim
    done = 0
    for n in sizes:
        kd, vd = (torch.from_numpy(rng.standard_normal((H, n - done, dim)).astype(np.float32)).cuda()
                  for _ in range(2))
        assert L.adaptq_mha_append_all_device(m, C.c_void_p(kd.data_ptr()),
                                              C.c_void_p(vd.data_ptr()), n - done, 0, None) == 0
        got = L.adaptq_ggml_attn_f32_device(m, C.c_void_p(qd.data_ptr()), dim, H, nq, row, H * row,
                                            C.c_void_p(od.data_ptr()), row, H * row, None)
        assert got == min(n, cap), err()
        y, k, v = od.cpu().numpy(), kd.cpu().numpy(), vd.cpu().numpy()
        for h, o in refs.items():
            for t in range(n - done):
                o.append(k[h, t], v[h, t], t)
            for j in (0, nq // 2, nq - 1):
                assert rel_err(y[j, h], o.compute(qs[j, h])[0]) <= 1e-4, (n, h, j)
        done = n
    L.adaptq_mha_destroy(m)


@pytest.mark.parametrize("vm,hyb,nq,kb", [(0.0, 0, 1, 4), (0.0, 0, 3, 4), (0.0, 0, 40, 4),
                                          (0.95, 0, 3, 4), (0.0, 512, 3, 4), (0.0, 0, 5, 16)])
@pytest.mark.parametrize("place", ["apart", "same", "shifted", "strided"])
def test_ggml_rows_in_place(oracle, vm, hyb, nq, kb, place):
    """The attention operator on rows that it reads and writes in place
    (packed, apart or the very same) and on rows that it must copy (a
    destination shifted into the queries, another stride)."""
    import torch
    H, dim, n = 3, 64, 300
    rng = np.random.default_rng(nq + kb)
    m = L.adaptq_mha_create(H, dim, kb, 4, 400, 9, vm, hyb)
    K = rng.standard_normal((H, n, dim)).astype(np.float32)
    V = rng.standard_normal((H, n, dim)).astype(np.float32)
    kd, vd = torch.from_numpy(K).cuda(), torch.from_numpy(V).cuda()
    assert L.adaptq_mha_append_all_device(m, C.c_void_p(kd.data_ptr()), C.c_void_p(vd.data_ptr()),
                                          n, 0, None) == 0
    q = rng.standard_normal((nq, H, dim)).astype(np.float32)
    row = dim * 4
    hs = row + 32 if place == "strided" else row       # between heads
    size = nq * H * hs // 4
    buf = torch.zeros(3 * size + 64, device="cuda")
    qv = buf[:size].view(nq, H, hs // 4)
    qv[:, :, :dim] = torch.from_numpy(q).cuda()
    at = {"apart": 2 * size, "same": 0, "shifted": 4, "strided": 2 * size}[place]
    got = L.adaptq_ggml_attn_f32_device(
        m, C.c_void_p(buf.data_ptr()), dim, H, nq, hs, H * hs,
        C.c_void_p(buf.data_ptr() + 4 * at), hs, H * hs, None)
    assert got == n
    y = buf[at:at + size].view(nq, H, hs // 4)[:, :, :dim].cpu().numpy()
    for h in range(H):
        o = oracle.head(dim, kb, 4, 400, I.mha_seed(9, h), vm, hyb)
        for t in range(n):
            o.append(K[h, t], V[h, t], t)
        for j in range(nq):
            assert rel_err(y[j, h], o.compute(q[j, h])[0]) <= 1e-4, (h, j)
    L.adaptq_mha_destroy(m)
