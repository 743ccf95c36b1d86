"""The append kernels above padded 128 (a wave per row, or per 2048 / padded
rows) against the oracle: codes, scales and the fp32 mirror's answers.

Bar: bit-exact rings; the mirror is read back through a decode, whose outputs
stay within the 1e-4 of every output test (fp32 rows, at most 24 tokens)."""
import ctypes as C

import numpy as np
import pytest

from adaptq_amd import _lib
from golden import inputs as I
from gpu_head import GpuHead, err, rel_err, same_bits

pytestmark = pytest.mark.gpu
L = _lib.lib


def _rows(rng, n, dim):
    """Normal rows with, among them, rows at the edges of the codec: zeros,
    single spikes, sums of squares around 1e-10, underflowing and overflowing
    squares, NaN and infinite entries."""
    x = rng.standard_normal((n, dim)).astype(np.float32)
    b = np.sqrt(1e-10 / dim)
    edge = [lambda r: r * 0, lambda r: r * np.float32(1e-20), lambda r: r * np.float32(3e-23),
            lambda r: r * np.float32(b * 0.999), lambda r: r * np.float32(b * 1.001),
            lambda r: r * np.float32(1e19), lambda r: np.where(np.arange(dim) == 7, r, 0),
            lambda r: np.where(np.arange(dim) == dim - 1, np.nan, r),
            lambda r: np.where(np.arange(dim) == 0, np.inf, r)]
    for i, t in enumerate(range(1, n, 5)):
        x[t] = edge[i % len(edge)](x[t])
    return x.astype(np.float32)


# (n per call, ...): one token; a few; whole wave groups and remainders of them;
# more than the ring holds (the call evicts its own first rows)
@pytest.mark.parametrize("dim,kb,vb,heads,cap,calls", [
    (256, 4, 2, 3, 40, (1, 1, 17, 1, 60)),
    (200, 3, 16, 2, 33, (1, 5, 1, 34)),
    (129, 2, 3, 2, 16, (1, 16, 1)),
    (512, 4, 3, 2, 24, (1, 9, 30)),
    (300, 16, 4, 2, 24, (1, 9, 30)),
    (1024, 2, 4, 2, 12, (1, 5, 20)),
    (1000, 3, 2, 2, 12, (1, 5, 20)),
    # many rows a call: several rows a wave (above 2,048 vectors)
    (256, 4, 2, 9, 950, (1000, 915)),
    (160, 3, 3, 9, 2000, (913, 914)),
    (512, 2, 4, 9, 950, (1001,)),
    (513, 4, 3, 9, 950, (917,)),
    (256, 16, 2, 9, 950, (1000,)),
    (1024, 4, 2, 5, 700, (513,)),
    (256, 4, 4, 300, 5, (16, 17)),  # a ring shorter than a wave's rows
])
def test_wide_append_bit_exact(oracle, torch_dev, dim, kb, vb, heads, cap, calls):
    print(f"wide append dim={dim} k{kb}v{vb} heads={heads} cap={cap} calls={calls}", flush=True)
    torch = torch_dev
    rng = np.random.default_rng(dim * 7 + kb + vb)
    seed = 99 + dim
    m = L.adaptq_mha_create(heads, dim, kb, vb, cap, seed, 0.0, 0)
    assert m, err()
    check = sorted({0, 1, heads // 2, heads - 1} & set(range(heads)))
    refs = {h: oracle.head(dim, kb, vb, cap, I.mha_seed(seed, h)) for h in check}
    for n in calls:
        K = np.stack([_rows(rng, n, dim) for _ in range(heads)])
        V = np.stack([_rows(rng, n, dim)[::-1] for _ in range(heads)])
        kd, vd = torch.from_numpy(K).cuda(), torch.from_numpy(V.copy()).cuda()
        assert L.adaptq_mha_append_all_device(m, C.c_void_p(kd.data_ptr()),
                                              C.c_void_p(vd.data_ptr()), n, 0, None) == 0, err()
        torch.cuda.synchronize()
        for h in check:
            for t in range(n):
                refs[h].append(K[h, t], V[h, t], t)
    for h in check:
        g = GpuHead.wrap(L.adaptq_mha_head(m, h), dim)
        oi = refs[h].info()
        assert (g.info()["head"], g.info()["size"]) == (oi["head"], oi["size"])
        for x, y, what in zip(g.read_slots(0, oi["size"]), refs[h].read_slots(0, oi["size"]),
                              ("k codes", "v codes", "k scale", "v scale")):
            assert same_bits(x, y), (h, what)
    L.adaptq_mha_destroy(m)


@pytest.mark.parametrize("dim,calls", [(256, (1, 1)), (200, (7, 1)), (1024, (1, 5)), (256, (20,)),
                                       (512, (24,))])
def test_wide_append_mirror(oracle, torch_dev, dim, calls):
    """The hybrid mirror's rows (up to 20 of them), through the hybrid branch;
    at 24 tokens the ring's own."""
    print(f"wide mirror dim={dim} calls={calls}", flush=True)
    torch = torch_dev
    heads, cap, hyb, seed = 500 if calls[0] >= 20 else 3, 64, 20, 5
    rng = np.random.default_rng(dim)
    m = L.adaptq_mha_create(heads, dim, 4, 2, cap, seed, 0.0, hyb)
    assert m, err()
    refs = [oracle.head(dim, 4, 2, cap, I.mha_seed(seed, h), 0.0, hyb) for h in range(3)]
    for n in calls:
        kd, vd = (torch.from_numpy(rng.standard_normal((heads, n, dim)).astype(np.float32)).cuda()
                  for _ in range(2))
        assert L.adaptq_mha_append_all_device(m, C.c_void_p(kd.data_ptr()),
                                              C.c_void_p(vd.data_ptr()), n, 0, None) == 0, err()
        for h, o in enumerate(refs):
            for t in range(n):
                o.append(kd[h, t].cpu().numpy(), vd[h, t].cpu().numpy(), t)
    q = rng.standard_normal((heads, dim)).astype(np.float32)
    out = np.zeros((heads, dim), np.float32)
    assert L.adaptq_mha_compute_all(m, _lib.fptr(q), _lib.fptr(out)) == sum(calls), err()
    for h, o in enumerate(refs):
        assert rel_err(out[h], o.compute(q[h])[0]) <= 1e-4, h
    L.adaptq_mha_destroy(m)
