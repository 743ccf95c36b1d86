"""The decode step over the fp32 mirror in one launch, and steps whose rows are
fp16 or bf16, against the oracle: ring bytes and scales bit-exact, outputs
within 1e-4 norm-wise (fp32 rows); half-precision steps give the fp32 step's
answer on the same values, rounded to nearest even, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from adaptq_amd import _lib
from golden import inputs as I
from gpu_head import GpuHead, err, rel_err, same_bits

pytestmark = pytest.mark.gpu
L = _lib.lib


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _step(m, k, v, q, o, io, t):
    n = L.adaptq_mha_step_device(m, _ptr(k), _ptr(v), _ptr(q), _ptr(o), io, t, None)
    assert n >= 0, err()
    return n


# steps: tokens fed; the mirror ends past hyb tokens and at the first eviction
@pytest.mark.parametrize("dim,kb,vb,cap,hyb,steps", [
    (64, 4, 4, 100, 70, 110), (64, 2, 3, 600, 512, 515), (48, 3, 2, 80, 66, 70),
    (128, 4, 2, 300, 130, 140), (80, 2, 4, 66, 512, 68), (128, 3, 16, 40, 20, 24),
    (256, 4, 2, 80, 65, 67), (200, 16, 4, 20, 30, 24), (33, 4, 4, 20, 30, 24),
    (512, 4, 4, 20, 10, 12), (32, 4, 4, 20, 10, 12),
])
def test_mirror_steps(oracle, torch_dev, dim, kb, vb, cap, hyb, steps):
    torch = torch_dev
    H, seed = 3, 40 + dim
    rng = np.random.default_rng(dim + steps)
    m = L.adaptq_mha_create(H, dim, kb, vb, cap, seed, 0.9, hyb)
    assert m, err()
    refs = [oracle.head(dim, kb, vb, cap, I.mha_seed(seed, h), 0.9, hyb) for h in range(H)]
    o = torch.empty(H, dim, device="cuda")
    for t in range(steps):
        k, v, q = (rng.standard_normal((H, dim)).astype(np.float32) for _ in range(3))
        if t % 7 == 3:
            k[0] = 0.0
            v[1] *= np.float32(1e-20)
        kd, vd, qd = (torch.from_numpy(x).cuda() for x in (k, v, q))
        if t == 9:
            n = L.adaptq_mha_append_compute_all_device(m, _ptr(kd), _ptr(vd), t, _ptr(qd),
                                                       _ptr(o), None)
        else:
            n = _step(m, kd, vd, qd, o, 0, t)
        assert n == min(t + 1, cap)
        y = o.cpu().numpy()
        for h, r in enumerate(refs):
            r.append(k[h], v[h], t)
            if t < 5 or t % 16 in (0, 15) or t > steps - 6:
                assert rel_err(y[h], r.compute(q[h])[0]) <= 1e-4, (t, h)
    for h, r in enumerate(refs):
        g = GpuHead.wrap(L.adaptq_mha_head(m, h), dim)
        oi = r.info()
        assert (g.info()["head"], g.info()["size"]) == (oi["head"], oi["size"])
        for x, y in zip(g.read_slots(0, oi["size"]), r.read_slots(0, oi["size"])):
            assert same_bits(x, y)
    L.adaptq_mha_destroy(m)


@pytest.mark.parametrize("dim,vm,hyb", [(64, 0.9, 20), (96, 0.9, 20), (64, 0.0, 0), (256, 0.0, 12)])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_half_rows(torch_dev, dim, vm, hyb, dtype):
    """Across the mirror's end into the sparse-V and dense branches, with large
    values and ones that underflow in the rows' type."""
    torch = torch_dev
    dt = getattr(torch, dtype)
    io = {"float16": 1, "bfloat16": 2}[dtype]
    H = 4
    a, b = (L.adaptq_mha_create(H, dim, 4, 4, 64, 3, vm, hyb) for _ in range(2))
    g = torch.Generator(device="cuda")
    g.manual_seed(dim)
    for t in range(40):
        x = torch.randn(3, H, dim, device="cuda", generator=g)
        x[1, 0] *= 1e-7 if t % 3 else 1e4  # (below fp16's 65,504)
        x = x.to(dt)
        o, o32 = torch.empty(H, dim, device="cuda", dtype=dt), torch.empty(H, dim, device="cuda")
        x32 = x.float()
        _step(a, x[0], x[1], x[2], o, io, t)
        _step(b, x32[0], x32[1], x32[2], o32, 0, t)
        assert torch.equal(o, o32.to(dt)), t
    assert L.adaptq_mha_step_device(a, _ptr(x), _ptr(x), _ptr(x), _ptr(x), 3, 0, None) == -1
    for m in (a, b):
        L.adaptq_mha_destroy(m)


def test_module_types(torch_dev):
    """The torch module on fp32, fp16, bf16 and float64 tensors, strided ones and
    mixed types among them: the output in q's type, as the step on fp32 values
    gives it."""
    torch = torch_dev
    from adaptq_amd import AdaptQAttention
    H, dim = 3, 64
    base = AdaptQAttention(dim, H)
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    for dt in (torch.float32, torch.float16, torch.bfloat16, torch.float64):
        mod = AdaptQAttention(dim, H)
        base.reset_cache()
        for t in range(6):
            x = torch.randn(3, 1, H, 2 * dim, device="cuda", generator=g).to(dt)
            q, k, v = (y[..., ::2] if t % 2 else y[..., :dim] for y in x)
            if t == 4:
                k = k.float()
            y = mod(q, k, v)
            ref = base(q.float(), k.float(), v.float())
            assert y.dtype == dt and y.shape == (1, H, dim) and torch.equal(y, ref.to(dt)), (dt, t)


@pytest.mark.parametrize("dim,vm,hyb", [(64, 0.0, 0), (128, 0.0, 0), (64, 0.9, 20)])
def test_half_rows_captured_first(torch_dev, dim, vm, hyb):
    """A half-precision step that no such step went before, captured: its
    conversions take no memory that is not there, and later calls on the MHA (the
    ggml operator's, on more and strided rows) leave that memory to the graph."""
    torch = torch_dev
    H, n, nq = 4, 20, 40
    a, b = (L.adaptq_mha_create(H, dim, 4, 4, 64, 3, vm, hyb) for _ in range(2))
    g = torch.Generator(device="cuda").manual_seed(dim)
    rows = torch.randn(2, H, n, dim, device="cuda", generator=g)
    x = torch.randn(3, H, dim, device="cuda", generator=g).half()
    for m in (a, b):
        assert L.adaptq_mha_append_all_device(m, _ptr(rows[0]), _ptr(rows[1]), n, 0, None) == 0
    torch.cuda.synchronize()
    want, got = (torch.zeros(H, dim, device="cuda", dtype=torch.float16) for _ in range(2))
    if vm:  # sparse-V needs a workspace: any decode of this branch leaves one
        for m in (a, b):
            f = x.float()
            _step(m, f[0], f[1], f[2], torch.empty_like(f[0]), 0, n)
        torch.cuda.synchronize()
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        r = L.adaptq_mha_step_device(a, _ptr(x[0]), _ptr(x[1]), _ptr(x[2]), _ptr(got), 1, n,
                                     C.c_void_p(s.cuda_stream))
    assert r > 0, err()
    q = torch.randn(nq, H, dim + 8, device="cuda", generator=g)
    o, row = torch.empty_like(q), 4 * (dim + 8)
    for m in (a, b):
        assert L.adaptq_ggml_attn_f32_device(m, _ptr(q), dim, H, nq, row, H * row, _ptr(o), row,
                                             H * row, None) >= 0, err()
    torch.cuda.synchronize()
    graph.replay()
    _step(b, x[0], x[1], x[2], want, 1, n)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    del graph
    for m in (a, b):
        L.adaptq_mha_destroy(m)


@pytest.mark.parametrize("place", ["keys", "vals", "same keys", "same vals", "same queries"])
@pytest.mark.parametrize("dtype", ["float32", "float16"])
def test_outputs_over_rows(torch_dev, place, dtype):
    """Outputs shifted into the step's keys or values (more heads than run at
    once, so that some would read rows that others have written over) or exactly on
    its rows."""
    torch = torch_dev
    dt, io = getattr(torch, dtype), 0 if dtype == "float32" else 1
    # (a multiple of 8 heads on: the same XCD, whose L2 shows it the writes)
    H, dim, shift = 2048, 64, 1504
    g = torch.Generator(device="cuda").manual_seed(3)
    first, x = (torch.randn(3, H, dim, device="cuda", generator=g).to(dt) for _ in range(2))
    want = torch.empty(H, dim, device="cuda", dtype=dt)
    at = ("keys", "vals", "queries").index(place.split()[-1])
    off = 0 if place.startswith("same") else shift * dim
    bufs = [torch.zeros(H + shift, dim, device="cuda", dtype=dt) for _ in range(3)]
    for b, r in zip(bufs, x):
        b[:H] = r
    out = bufs[at].view(-1)[off:off + H * dim]
    for rows, o in ((x, want), (bufs, out)):
        m = L.adaptq_mha_create(H, dim, 4, 4, 8, 5, 0.0, 8)
        assert m, err()
        _step(m, *first, torch.empty_like(want), io, 0)
        _step(m, *rows, o, io, 1)
        torch.cuda.synchronize()
        L.adaptq_mha_destroy(m)
    assert torch.equal(out.view(H, dim), want)


def test_captured_step_past_the_kernel(torch_dev):
    """A step captured at 510 tokens and replayed past the 512 that its launch
    covers: those 512, the oldest, keep their softmax."""
    torch = torch_dev
    H, dim, n, replays = 3, 64, 509, 12
    g = torch.Generator(device="cuda").manual_seed(8)
    rows = torch.randn(2, H, n, dim, device="cuda", generator=g)
    x = torch.randn(3, H, dim, device="cuda", generator=g)
    out = torch.zeros(H, dim, device="cuda")
    m = L.adaptq_mha_create(H, dim, 4, 4, 1000, 3, 0.0, 600)
    assert L.adaptq_mha_append_all_device(m, _ptr(rows[0]), _ptr(rows[1]), n, 0, None) == 0, err()
    torch.cuda.synchronize()
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        r = L.adaptq_mha_step_device(m, _ptr(x[0]), _ptr(x[1]), _ptr(x[2]), _ptr(out), 0, n,
                                     C.c_void_p(s.cuda_stream))
    assert r == n + 1, err()
    for i in range(1, replays + 1):
        graph.replay()
        torch.cuda.synchronize()
        c = min(i, 512 - n)
        k, v = (torch.cat((old, new[:, None].expand(H, c, dim)), 1).double().cpu()
                for old, new in ((rows[0], x[0]), (rows[1], x[1])))
        w = torch.softmax((k * x[2].double().cpu()[:, None]).sum(2) / dim ** 0.5, 1)
        assert rel_err(out.cpu(), (w[:, :, None] * v).sum(1)) <= 1e-5, i
    del graph
    L.adaptq_mha_destroy(m)
