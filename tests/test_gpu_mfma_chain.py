"""v_mfma_f32_16x16x4 adds its four products to an entry one after another, each
a fused multiply-add rounded as fmaf: the many-query decode (mquery.hip) takes a
chain of it for the reference's chain of fmaf.  Bit for bit with fmaf on the
device, and with a chain in 64 bits rounded once a step where that is exact."""
import ctypes as C
import os

import numpy as np
import pytest

from adaptq_amd.build import PROBE_LIB

pytestmark = pytest.mark.gpu

BOOK = np.array([-2.4008, -1.8944, -1.5105, -1.2016, -0.9138, -0.6402, -0.3795, -0.1258], np.float32)


def _operands(kind, n, K, rng):
    a, b = (rng.standard_normal((n, 16, K)).astype(np.float32) for _ in range(2))
    c = rng.standard_normal((n, 16, 16)).astype(np.float32)
    if kind == "codes":  # a decode's own: codebook values and rotated queries, from 0
        a = np.concatenate((BOOK, -BOOK))[rng.integers(0, 16, a.shape)]
        b *= np.float32(8.0)
        c[:] = 0.0
    elif kind == "spread":  # exponents over the whole range of products
        b = np.ldexp(b, rng.integers(-60, 60, b.shape)).astype(np.float32)
        a = np.ldexp(a, rng.integers(-60, 60, a.shape)).astype(np.float32)
    elif kind == "denormal":  # products and sums below 2^-126, some operands too
        a = np.ldexp(a, rng.integers(-146, -60, a.shape)).astype(np.float32)
        b = np.ldexp(b, rng.integers(-70, 1, b.shape)).astype(np.float32)
        c = np.ldexp(c, -140).astype(np.float32)
    elif kind == "large":  # up to overflow
        a = np.ldexp(a, rng.integers(50, 64, a.shape)).astype(np.float32)
        b = np.ldexp(b, rng.integers(50, 63, b.shape)).astype(np.float32)
    elif kind == "zeros":
        a[rng.random(a.shape) < 0.5] = -0.0
        b[rng.random(b.shape) < 0.5] = 0.0
        c[:] = -0.0
    elif kind == "cancel":  # sums that nearly vanish
        a[:, :, 1::2] = -a[:, :, 0::2]
        b[:, :, 1::2] = b[:, :, 0::2] * np.float32(1 + 2.0 ** -22)
    return a, b.transpose(0, 2, 1).copy(), c


@pytest.mark.parametrize("kind", ["plain", "codes", "spread", "denormal", "large", "zeros", "cancel"])
@pytest.mark.parametrize("K", [4, 8, 16, 128])
def test_chain(torch_dev, kind, K):
    torch = torch_dev
    lib = C.CDLL(PROBE_LIB)
    n = 64
    rng = np.random.default_rng(K)
    a, b, c = _operands(kind, n, K, rng)
    ad, bd, cd = (torch.from_numpy(x).cuda() for x in (a, b, c))
    m, f = torch.zeros_like(cd), torch.zeros_like(cd)
    p = [C.c_void_p(t.data_ptr()) for t in (ad, bd, cd, m, f)]
    assert lib.adaptq_probe_chain(*p, n, K, None) == 0
    torch.cuda.synchronize()
    m, f = m.cpu().numpy(), f.cpu().numpy()
    both_nan = np.isnan(m) & np.isnan(f)
    diff = (m.view(np.uint32) != f.view(np.uint32)) & ~both_nan
    assert not diff.any(), (kind, K, m[diff][:4], f[diff][:4])
    if kind in ("plain", "codes"):
        # the device's fmaf is one: products of 24-bit values are exact in 64 bits,
        # and so is their sum with the entry unless exponents lie 28 apart
        acc = c.astype(np.float64)
        for k in range(K):
            acc = (a[:, :, k, None].astype(np.float64) * b[:, None, k].astype(np.float64)
                   + acc).astype(np.float32).astype(np.float64)
        odd = np.count_nonzero(acc.astype(np.float32).view(np.uint32) != f.view(np.uint32))
        assert odd <= 1e-4 * f.size  # double rounding


def test_refused_sizes():
    lib = C.CDLL(PROBE_LIB)
    one = C.c_void_p(16)
    for n, K in ((0, 4), (1, 0), (1, 6), (1, 8192), ((1 << 20) + 1, 4)):
        assert lib.adaptq_probe_chain(one, one, one, one, one, n, K, None) == -1
    assert lib.adaptq_probe_chain(None, one, one, one, one, 1, 4, None) == -1
