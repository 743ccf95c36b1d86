"""Zero probabilities in the sparse-V selection: they are taken oldest first,
as any equal ones.  Which of them are selected shows where a V row's scale is
not finite (an overflowed activation): its weight is 0 times that scale, NaN,
and so is the output.  Per-token weights bit for bit with the oracle's (a NaN
equals a NaN), at 1, 2, 4 and 8 tokens a thread and above the in-LDS sort."""
import ctypes as C

import numpy as np
import pytest

from adaptq_amd import _lib
from gpu_head import GpuHead, err, rel_err
from test_gpu_sparse_select import gpu_weights

pytestmark = pytest.mark.gpu
L = _lib.lib

SIZES = [63, 1000, 1023, 1999, 2048, 2999, 3500, 7001, 8192, 9000]


def _rows(rng, dim, n, tops, q):
    """K rows of which only ``tops`` keep a probability that is not zero (equal
    ones: the rest lie 200 below), and N(0,1) V rows."""
    K = (0.1 * rng.standard_normal((n, dim))).astype(np.float32)
    K[tops] = 8.0 * q / np.linalg.norm(q)
    return K, rng.standard_normal((n, dim)).astype(np.float32)


def _poison(V, rows):
    """Rows whose scale is inf (squares that overflow, an inf) or NaN."""
    rows = np.asarray(rows)
    V[rows[0::3]] = 1e20
    V[rows[1::3], 5] = np.nan
    V[rows[2::3], 7] = np.inf


def _check(oracle, dim, n, v_mass, K, V, q, label):
    g = GpuHead(dim, 4, 2, n, 7, v_mass, 0)
    o = oracle.head(dim, 4, 2, n, 7, v_mass, 0)
    for t in range(n):
        g.append(K[t], V[t], t)
        o.append(K[t], V[t], t)
    wo, r = o.sparse_weights(q), o.compute(q)[0]
    for _ in range(3):  # the order must not depend on which wave comes first
        wg = gpu_weights(g, q, n)
        bad = np.flatnonzero(np.isnan(wg) != np.isnan(wo))
        assert bad.size == 0, (label, bad[:8], wg[bad[:8]], wo[bad[:8]])
        fin = ~np.isnan(wo)
        assert np.array_equal(wg[fin].view(np.uint32), wo[fin].view(np.uint32)), label
        y = g.compute(q)[0]
        assert np.array_equal(np.isfinite(y), np.isfinite(r)), label
        if np.isfinite(r).all():
            assert rel_err(y, r) <= 1e-4, label
    return wo


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("m", [1, 2, 5])
def test_cut_inside_the_zeros(oracle, dim, n, m):
    """m equal probabilities at the ring's end, the last quad filled up with the
    oldest zeros: every other zero's V row is poisoned, then those alone."""
    rng = np.random.default_rng(1000 * dim + n + m)
    q = (30.0 * rng.standard_normal(dim)).astype(np.float32)
    tops = np.arange(n - m, n)
    fill = -m % 4  # zeros that complete the last quad
    K, V = _rows(rng, dim, n, tops, q)
    one = V.copy()
    _poison(one, np.arange(fill, n - m))
    w = _check(oracle, dim, n, 0.95, K, one, q, f"d{dim} n {n} m {m}: the others")
    assert np.isfinite(w).all() and (w != 0).sum() == m
    _poison(V, np.arange(fill))
    w = _check(oracle, dim, n, 0.95, K, V, q, f"d{dim} n {n} m {m}: the oldest")
    assert np.isnan(w).sum() == fill


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("n", SIZES)
def test_mass_never_reached(oracle, dim, n):
    """Every token is selected: no poisoned row may be left out."""
    rng = np.random.default_rng(dim + n)
    q = (30.0 * rng.standard_normal(dim)).astype(np.float32)
    K, V = _rows(rng, dim, n, np.arange(n // 2, n // 2 + 3), q)
    at = np.arange(0, n, 7)
    _poison(V, at)
    w = _check(oracle, dim, n, 2.0, K, V, q, f"d{dim} n {n} all")
    assert np.isnan(w).sum() >= at.size - 3


@pytest.mark.parametrize("dim,n", [(64, 700), (64, 2048), (64, 3000), (128, 2048), (128, 3000)])
def test_more_items_than_cus(torch_dev, dim, n):
    """The instances that share a CU: no poisoned zero reaches the output."""
    torch = torch_dev
    H = 300
    rng = np.random.default_rng(dim + n)
    q = (30.0 * rng.standard_normal(dim)).astype(np.float32)
    K, V = _rows(rng, dim, n, np.arange(n - 1, n), q)
    _poison(V, np.arange(3, n - 1))
    hs = [L.adaptq_create(dim, 4, 2, n, i, 0.95, 0) for i in range(H)]
    p = L.adaptq_plan_create((C.c_void_p * H)(*hs), H)
    assert p, err()
    k, v = (torch.from_numpy(x).cuda().expand(H, n, dim).contiguous() for x in (K, V))
    qd = torch.from_numpy(q).cuda().expand(H, dim).contiguous()
    o = torch.empty_like(qd)
    assert L.adaptq_plan_append_device(p, C.c_void_p(k.data_ptr()), C.c_void_p(v.data_ptr()), n, 0,
                                       None) == 0, err()
    assert L.adaptq_plan_compute_device(p, C.c_void_p(qd.data_ptr()), C.c_void_p(o.data_ptr()),
                                        None) == 0, err()
    assert torch.isfinite(o).all()
    L.adaptq_plan_destroy(p)
    for h in hs:
        L.adaptq_destroy(h)
