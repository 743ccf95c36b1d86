"""The bucket sort of the sparse-V selection where it can go wrong: thread and
bucket counts' edges, probabilities that underflow to zero or are subnormal,
equal ones within and beyond a bucket's limit.  Per-token weights bit for bit
with the oracle's, as in test_gpu_sparse_select.py; and more items than CUs,
whose selection shares a CU with another's, against the same contexts one by
one (bit for bit: the V sums' order is the same) and against the oracle."""
import ctypes as C

import numpy as np
import pytest

from adaptq_amd import _lib
from gpu_head import GpuHead, err, rel_err
from test_gpu_sparse_select import check_selection

pytestmark = pytest.mark.gpu
L = _lib.lib


def _pair(oracle, dim, n, v_mass, rng, groups=None):
    g = GpuHead(dim, 4, 2, n, 7, v_mass, 0)
    o = oracle.head(dim, 4, 2, n, 7, v_mass, 0)
    base = rng.standard_normal((groups or n, dim)).astype(np.float32)
    K = base[np.arange(n) % len(base)]
    V = rng.standard_normal((n, dim)).astype(np.float32)
    for t in range(n):
        g.append(K[t], V[t], t)
        o.append(K[t], V[t], t)
    return g, o


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 3072, 3073,
                               4096, 4097, 8191, 8192])
def test_edges(oracle, dim, n):
    """Plain queries, ones so long that most probabilities underflow, and a
    short one whose probabilities are nearly equal."""
    rng = np.random.default_rng(n)
    g, o = _pair(oracle, dim, n, 0.95, rng)
    q = rng.standard_normal(dim).astype(np.float32)
    for scale in (1.0, 18.0, 70.0, 1e-4):
        check_selection(g, o, (q * np.float32(scale)).astype(np.float32), f"n {n} scale {scale}")


@pytest.mark.parametrize("n,groups", [(2000, 3), (2000, 5), (2000, 40), (3000, 1), (3000, 7),
                                      (8000, 15), (8000, 17), (8000, 900)])
@pytest.mark.parametrize("scale", [1.0, 25.0])
def test_ties(oracle, n, groups, scale):
    """Keys repeated so that a bucket holds equal probabilities below its limit
    and above it; at 25 some groups are subnormal, some zero."""
    rng = np.random.default_rng(n + groups)
    g, o = _pair(oracle, 64, n, 0.97, rng, groups)
    check_selection(g, o, (rng.standard_normal(64) * scale).astype(np.float32), f"{n} {groups}")


def test_mass_of_everything(oracle):
    """A mass the probabilities cannot reach takes every token, the zeros too."""
    rng = np.random.default_rng(5)
    g, o = _pair(oracle, 64, 1500, 2.0, rng)
    check_selection(g, o, (rng.standard_normal(64) * 30).astype(np.float32), "all")


@pytest.mark.parametrize("dim,kb,vb,n", [(64, 4, 2, 2048), (64, 3, 3, 2600), (64, 2, 4, 700),
                                         (128, 4, 4, 2049), (128, 3, 2, 1000)])
def test_more_items_than_cus(oracle, torch_dev, dim, kb, vb, n):
    torch = torch_dev
    H = 300
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    hs = [L.adaptq_create(dim, kb, vb, n, i, 0.95, 0) for i in range(H)]
    p = L.adaptq_plan_create((C.c_void_p * H)(*hs), H)
    assert p, err()
    k, v = (torch.randn(H, n, dim, device="cuda", generator=g) for _ in range(2))
    q = torch.randn(H, dim, device="cuda", generator=g)
    assert L.adaptq_plan_append_device(p, C.c_void_p(k.data_ptr()), C.c_void_p(v.data_ptr()), n, 0,
                                       None) == 0
    o = torch.empty_like(q)
    for _ in range(2):
        assert L.adaptq_plan_compute_device(p, C.c_void_p(q.data_ptr()), C.c_void_p(o.data_ptr()),
                                            None) == 0, err()
    y = o.cpu().numpy()
    for h in (0, 1, 150, H - 1):
        one = np.empty(dim, np.float32)
        qh = q[h].cpu().numpy()
        assert L.adaptq_compute(hs[h], _lib.fptr(qh), _lib.fptr(one)) == n
        assert np.array_equal(one.view(np.uint32), y[h].view(np.uint32)), h
        if h in (1, H - 1):
            r = oracle.head(dim, kb, vb, n, h, 0.95, 0)
            kh, vh = k[h].cpu().numpy(), v[h].cpu().numpy()
            for t in range(n):
                r.append(kh[t], vh[t], t)
            assert rel_err(y[h], r.compute(qh)[0]) <= 1e-4, h
    L.adaptq_plan_destroy(p)
    for h in hs:
        L.adaptq_destroy(h)
