"""Decode of many queries per head against the oracle, query by query: outputs
within 1e-4 norm-wise.  Through adaptq_compute_batch (one head) and the ggml
multi-query operator (every head of an MHA, queries [query][head][dim]); every
K/V bit width, padded 64 and 128 (one unpadded dim), query counts that leave
partial 16-query groups, a wrapped ring, and config 2's x20 outlier channels.
The short rings take the LUT kernel, one item a query; ``matrix`` cases have the
sizes at which the matrix-core kernel (mquery.hip: both products on fp32 MFMA,
the logits in the reference's own order) takes over, which they assert."""
import ctypes as C

import numpy as np
import pytest

import mq_rule
from adaptq_amd import _lib
from golden import inputs as I
from gpu_head import GpuHead, err, rel_err

pytestmark = pytest.mark.gpu
L = _lib.lib
TOL = 1e-4


@pytest.mark.parametrize("dim,kb,vb,cap,n,nq", [
    (128, 4, 4, 3000, 3000, 64), (64, 4, 2, 2100, 2100, 16), (128, 2, 3, 1000, 1000, 20),
    (64, 3, 3, 700, 700, 33), (128, 3, 2, 5000, 5000, 17), (64, 2, 4, 64, 64, 16),
    (96, 4, 2, 1500, 1500, 40), (128, 4, 4, 1024, 1500, 24), (64, 4, 3, 9000, 9000, 100),
])
def test_compute_batch_many_queries(oracle, dim, kb, vb, cap, n, nq):
    check_batch(oracle, dim, kb, vb, cap, n, nq)


@pytest.mark.parametrize("dim,kb,vb,cap,n,nq", [
    (128, 4, 4, 9400, 9400, 64), (64, 4, 2, 18700, 18700, 64), (96, 3, 2, 10000, 12345, 70),
    (50, 2, 3, 22000, 22000, 61),
])
def test_compute_batch_matrix(oracle, dim, kb, vb, cap, n, nq):
    assert mq_rule.takes(1, nq, min(n, cap), 64 if dim <= 64 else 128)
    check_batch(oracle, dim, kb, vb, cap, n, nq)


def check_batch(oracle, dim, kb, vb, cap, n, nq):
    print(f"multi-query d{dim} K{kb}V{vb} cap {cap} n {n} nq {nq}", flush=True)
    rng = np.random.default_rng(dim * 7 + n + nq)
    seed = int(rng.integers(0, 2**63))
    g = GpuHead(dim, kb, vb, cap, seed)
    o = oracle.head(dim, kb, vb, cap, seed)
    K = rng.standard_normal((n, dim)).astype(np.float32)
    V = rng.standard_normal((n, dim)).astype(np.float32)
    for t in range(n):
        g.append(K[t], V[t], t)
        o.append(K[t], V[t], t)
    qs = (rng.standard_normal((nq, dim)) * 1.5).astype(np.float32)
    ys, ng = g.compute_batch(qs)
    assert ng == min(n, cap)
    worst = 0.0
    for j in range(nq):
        r, _ = o.compute(qs[j])
        worst = max(worst, rel_err(ys[j], r))
    print(f"  worst norm-wise error over {nq} queries: {worst:.2e}", flush=True)
    assert worst <= TOL


def test_outlier_channels_many_queries(oracle):
    """Config 2's layer shape (d64 K4/V2, 512 tokens) with channels 3 and 17
    of K, V and the queries scaled x20: peaked softmaxes (logits of +-300),
    where one fp32 unit of a logit moves the outputs by ~3e-5, so only the
    reference's own rounding of the dot stays within the bar (a
    double-precision dot lands 1.3e-4 away)."""
    rng = np.random.default_rng(2)
    dim, n, nq = 64, 512, 48
    K = rng.standard_normal((n, dim)).astype(np.float32)
    V = rng.standard_normal((n, dim)).astype(np.float32)
    qs = rng.standard_normal((nq, dim)).astype(np.float32)
    for x in (K, V, qs):
        x[:, [3, 17]] *= 20.0
    seed = 42 ^ 5
    g = GpuHead(dim, 4, 2, n, seed)
    o = oracle.head(dim, 4, 2, n, seed)
    for t in range(n):
        g.append(K[t], V[t], t)
        o.append(K[t], V[t], t)
    ys, _ = g.compute_batch(qs)
    worst = max(rel_err(ys[j], o.compute(qs[j])[0]) for j in range(nq))
    # the same queries one at a time (the single-query LUT kernel)
    worst1 = max(rel_err(g.compute(qs[j])[0], o.compute(qs[j])[0]) for j in range(nq))
    print(f"outlier channels: worst norm-wise error {worst:.2e} batched, {worst1:.2e} one by one",
          flush=True)
    assert worst <= TOL and worst1 <= TOL


@pytest.mark.parametrize("dim,kb,vb,nq", [(64, 4, 2, 48), (128, 4, 4, 32), (128, 3, 3, 17)])
def test_outlier_channels_matrix(oracle, dim, kb, vb, nq):
    """The same peaked softmaxes through the matrix-core kernel: as many heads
    over 512 tokens as take it, through the ggml operator."""
    import torch
    n = 512
    H = mq_rule.heads_for(nq, n, dim)
    rng = np.random.default_rng(dim + nq)
    K, V = (rng.standard_normal((H, n, dim)).astype(np.float32) for _ in range(2))
    qs = rng.standard_normal((nq, H, dim)).astype(np.float32)
    for x in (K, V, qs):
        x[:, :, [3, 17]] *= 20.0
    m = L.adaptq_mha_create(H, dim, kb, vb, n, 42, 0.0, 0)
    assert m, err()
    kd, vd, qd = (torch.from_numpy(x).cuda() for x in (K, V, qs))
    od, row = torch.empty_like(qd), 4 * dim
    assert L.adaptq_mha_append_all_device(m, C.c_void_p(kd.data_ptr()), C.c_void_p(vd.data_ptr()),
                                          n, 0, None) == 0, err()
    assert L.adaptq_ggml_attn_f32_device(m, C.c_void_p(qd.data_ptr()), dim, H, nq, row, H * row,
                                         C.c_void_p(od.data_ptr()), row, H * row, None) == n, err()
    y = od.cpu().numpy()
    worst = 0.0
    for h in (0, 1, H // 2, H - 1):
        o = oracle.head(dim, kb, vb, n, I.mha_seed(42, h))
        for t in range(n):
            o.append(K[h, t], V[h, t], t)
        worst = max([worst] + [rel_err(y[j, h], o.compute(qs[j, h])[0]) for j in range(nq)])
    print(f"outlier channels, matrix cores: worst norm-wise error {worst:.2e}", flush=True)
    assert worst <= TOL
    L.adaptq_mha_destroy(m)


@pytest.mark.parametrize("H", [6, 8])
def test_ggml_multi_query_device(oracle, H):
    """Every head of an MHA, 32 queries each, through the ggml device
    operator (queries [query][head][dim] with padded strides); 6 heads take
    the LUT kernel, 8 the matrix cores."""
    import torch
    dim, kb, vb, n, nq = 128, 4, 2, 2500, 32
    assert mq_rule.takes(H, nq, n, dim) == (H == 8)
    rng = np.random.default_rng(9)
    m = L.adaptq_mha_create(H, dim, kb, vb, 4096, 77, 0.0, 0)
    assert m, err()
    K = rng.standard_normal((n, H, dim)).astype(np.float32)
    V = rng.standard_normal((n, H, dim)).astype(np.float32)
    for t in range(n):
        assert L.adaptq_mha_append_all(m, _lib.fptr(K[t]), _lib.fptr(V[t]), t) == 0, err()
    row, hstride = dim * 4, (dim + 8) * 4  # padded head stride
    qh = np.zeros((nq, H, dim + 8), np.float32)
    qh[:, :, :dim] = rng.standard_normal((nq, H, dim))
    qd = torch.from_numpy(qh).cuda()
    od = torch.zeros(nq, H, dim + 8, device="cuda")
    got = L.adaptq_ggml_attn_f32_device(m, C.c_void_p(qd.data_ptr()), dim, H, nq, hstride,
                                        H * hstride, C.c_void_p(od.data_ptr()), hstride,
                                        H * hstride, None)
    assert got == n, err()
    y = od.cpu().numpy()
    assert not y[:, :, dim:].any()  # padding untouched
    worst = 0.0
    for h in range(H):
        o = oracle.head(dim, kb, vb, 4096, I.mha_seed(77, h))
        for t in range(n):
            o.append(K[t, h], V[t, h], t)
        for j in range(nq):
            worst = max(worst, rel_err(y[j, h, :dim], o.compute(qh[j, h, :dim])[0]))
    print(f"ggml multi-query: worst norm-wise error {worst:.2e}", flush=True)
    assert worst <= TOL
    L.adaptq_mha_destroy(m)
