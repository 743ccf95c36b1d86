"""The calls that programs make of this library, with the sizes they make them at.

A case is one kind of call on one shape:

  session  the torch module, one token at a time from an empty cache
  engine   one decode step through the numpy Engine (host arrays in and out)
  layers   one decode step of a stack of layers, one call a layer
  plan     one decode step of many contexts in one launch each
  queries  many queries over one layer's cache (the ggml attention operator)
  prefill  a prompt appended in bulk, then the first decode on it

``listed`` holds the sizes of the repository's own configurations and tests and
what lies between them, ``draw`` more of the same ranges.  ``exact`` restates
the cache format (signs, Hadamard rotation, codebooks, scales) in torch with the
32-bit roundings that define the codes, and computes the attention over the
dequantised rows in 64 bits.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

U64 = (1 << 64) - 1
CODEBOOK = {
    2: (-1.5104, -0.4528, 0.4528, 1.5104),
    3: (-2.1529, -1.3439, -0.7560, -0.2451, 0.2451, 0.7560, 1.3439, 2.1529),
    4: (-2.4008, -1.8944, -1.5105, -1.2016, -0.9138, -0.6402, -0.3795, -0.1258,
        0.1258, 0.3795, 0.6402, 0.9138, 1.2016, 1.5105, 1.8944, 2.4008),
}
CHUNK = 1 << 30  # values of K drawn at once


def _case(kind, **kw):
    c = dict(kind=kind, sequences=1, layers=1, heads=8, dim=128, k_bits=4, v_bits=4,
             first_k_bits=0, tokens=1024, least=0, capacity=1024, v_mass=0.0, hybrid=0,
             append=1, queries=1, values="normal", dtype="float32")
    c.update(kw)
    return c


def listed():
    return [
        # a chat's first tokens through the torch module, as a generation loop
        # feeds them: half-precision tensors on the GPU, the module's defaults
        # (fp32 mirror up to 512 tokens)
        _case("session", name="module_session_64", heads=14, dim=64, tokens=64, capacity=4096,
              v_mass=0.95, hybrid=512, append=64, dtype="float16"),
        # the Engine's decode step under its defaults on a full small cache:
        # numpy in, numpy out, sparse-V
        _case("engine", name="engine_step_2048", heads=4, dim=64, k_bits=4, v_bits=2,
              tokens=2048, capacity=2048, v_mass=0.95, hybrid=512),
        # a 22-layer model's decode step, a call a layer: heavy-tailed values,
        # fp32 keys in layer 0, 3-bit keys after it
        _case("layers", name="layers_step_1280", layers=22, heads=4, dim=64, k_bits=3, v_bits=2,
              first_k_bits=16, tokens=1280, capacity=1280, values="student"),
        # a 24-layer model's decode step in one launch, the Engine's default
        # sparse-V over 2,048 tokens
        _case("plan", name="plan_sparse_2048", layers=24, heads=14, dim=64, k_bits=4, v_bits=2,
              tokens=2048, capacity=2048, v_mass=0.95, hybrid=512),
        # sequences of uneven length decoded together, as a server batches
        # them; a head dimension that is no power of two, 3-bit codes
        _case("plan", name="plan_ragged_d96", sequences=16, layers=4, heads=8, dim=96, k_bits=3,
              v_bits=3, tokens=8192, least=256, capacity=8192, append=0),
        # wide heads
        _case("plan", name="plan_d256_4096", sequences=8, layers=4, heads=8, dim=256, k_bits=4,
              v_bits=2, tokens=4096, capacity=4096),
        # one layer with a long ring: a decode step with every token weighed ...
        _case("layers", name="long_step_32768", tokens=32768, capacity=32768),
        # ... and the same under the default sparse-V
        _case("layers", name="long_sparse_32768", tokens=32768, capacity=32768, v_mass=0.95,
              hybrid=512),
        # many queries over the same ring (speculation, scoring, a prompt's tail)
        _case("queries", name="long_queries_64", tokens=32768, capacity=32768, queries=64,
              append=0),
        # a prompt longer than the ring, then its first decode
        _case("prefill", name="long_prefill_40000", tokens=0, capacity=32768, append=40000),
        # a batch of prompts, then the first decode on them
        _case("prefill", name="batch_prefill_8192", sequences=4, layers=32, v_bits=2, tokens=0,
              capacity=8192, append=8192),
        # the decode step of 64 sequences x 32 layers x 8 heads in one launch
        _case("plan", name="batch_decode_8192", sequences=64, layers=32, v_bits=2, tokens=8192,
              capacity=8192, append=0),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("session", "engine", "layers", "layers", "plan", "plan", "plan", "queries",
                       "prefill", "prefill"))
    dim = rng.choice((64, 64, 80, 96, 128, 128))
    k_bits, v_bits = rng.choice(((4, 2), (4, 2), (4, 4), (3, 2), (3, 3), (2, 2), (3, 4)))
    values = rng.choice(("normal", "normal", "student", "outliers"))
    v_mass = rng.choice((0.0, 0.95))
    c = dict(dim=dim, k_bits=k_bits, v_bits=v_bits, values=values)
    if kind == "session":
        n = _spread(rng, 8, 256)
        return _case(kind, **{**c, "heads": rng.randint(2, 16), "tokens": n, "append": n,
                              "capacity": 4096, "v_mass": 0.95, "hybrid": 512,
                              "dtype": rng.choice(("float16", "float32"))})
    if kind == "engine":
        n = _spread(rng, 256, 8192)
        return _case(kind, **{**c, "heads": rng.randint(2, 16), "tokens": n, "capacity": n,
                              "v_mass": 0.95, "hybrid": 512})
    if kind == "layers":
        n = _spread(rng, 128, 32768)
        layers = rng.randint(1, 4) if n > 4096 else rng.randint(4, 32)
        return _case(kind, **{**c, "layers": layers, "heads": rng.randint(2, 16), "tokens": n,
                              "capacity": n, "v_mass": v_mass,
                              "first_k_bits": rng.choice((0, 16))})
    if kind == "plan":
        if rng.random() < 0.25:  # wide heads
            n = _spread(rng, 256, 8192)
            units = _spread(rng, 1, 64)
            return _case(kind, **{**c, "dim": rng.choice((160, 192, 256)), "layers": units,
                                  "tokens": n, "capacity": n})
        n = _spread(rng, 256, 8192)
        heads = rng.randint(4, 16)
        sequences, layers = _spread(rng, 1, 32), rng.randint(1, 32)
        while sequences * layers * heads * n * dim > 1 << 31:
            sequences, layers = max(1, sequences // 2), max(1, layers * 3 // 4)
        if n <= 512 and rng.random() < 0.5:  # the fp32 mirror
            return _case(kind, **{**c, "sequences": sequences, "layers": layers, "heads": heads,
                                  "tokens": n, "capacity": n, "v_mass": 0.95, "hybrid": 512,
                                  "append": 0})
        if n >= 1024 and sequences > 1 and rng.random() < 0.5:
            return _case(kind, **{**c, "sequences": sequences, "layers": layers, "heads": heads,
                                  "tokens": n, "least": n // 32, "capacity": n,
                                  "v_mass": v_mass, "append": 0})
        return _case(kind, **{**c, "sequences": sequences, "layers": layers, "heads": heads,
                              "tokens": n, "capacity": n, "v_mass": v_mass})
    if kind == "queries":
        n = _spread(rng, 512, 32768)
        return _case(kind, **{**c, "heads": rng.randint(2, 16), "tokens": n, "capacity": n,
                              "queries": _spread(rng, 2, 96), "append": 0})
    n, heads = _spread(rng, 64, 40000), rng.randint(4, 16)
    layers = max(1, min(_spread(rng, 1, 64), (1 << 30) // (n * heads * dim)))
    return _case("prefill", **{**c, "layers": layers, "heads": heads, "tokens": 0,
                               "append": n, "capacity": rng.choice((n, max(64, n * 3 // 4)))})


# ---------------------------------------------------------------- the shapes

def _lengths(c):
    """Cached tokens of each sequence: all alike, or spread over the logarithm
    between ``least`` and ``tokens``."""
    if not c["least"]:
        return [c["tokens"]] * c["sequences"]
    lo, hi = c["least"], c["tokens"]
    return [int(lo * (hi / lo) ** ((0.618 * (i + 1)) % 1.0)) for i in range(c["sequences"])]


def _bits_of(c, layer):
    return c["first_k_bits"] if c["first_k_bits"] and layer == 0 else c["k_bits"]


def _padded(dim):
    return 1 << (dim - 1).bit_length()


def _row_bytes(p, bits):
    return 4 * p if bits == 16 else p * bits // 8


def work(c):
    p, heads, dim = _padded(c["dim"]), c["heads"], c["dim"]
    rows = nbytes = 0
    for n in _lengths(c):
        for layer in range(c["layers"]):
            kb = _bits_of(c, layer)
            row = _row_bytes(p, kb) + _row_bytes(p, c["v_bits"]) + 8
            if c["kind"] == "session":  # fp32 rows; token t attends over t + 1
                n_read = c["append"] * (c["append"] + 1) // 2
                rows += heads * n_read
                nbytes += heads * (n_read * 8 * dim + c["append"] * (16 * dim + row))
                continue
            n = min(n + c["append"], c["capacity"])
            if c["hybrid"] >= n and c["tokens"] + c["append"] <= c["capacity"]:
                nbytes += heads * n * 8 * dim
            else:
                nbytes += heads * n * row
            kept = min(c["append"], c["capacity"])  # rows read, coded and written
            nbytes += heads * kept * (8 * dim + row) + heads * c["queries"] * 8 * dim
            rows += heads * n * c["queries"]
    return {"bytes": float(nbytes), "flops": float(4 * p * rows)}


def tolerance(c):
    if c["dtype"] == "float16":
        return {"rel": 1e-3}  # the answers are rounded to 11 bits
    if c["kind"] != "session" and c["v_mass"] > 0 and c["k_bits"] != 16:
        # which tokens lie inside the mass depends on the last bits of 32-bit
        # sums over up to 32,768 tokens; one token more or less at the cut
        return {"rel": 3e-3}
    if c["values"] == "outliers":
        return {"rel": 1e-4}  # logits in the hundreds: their last bit is 1e-5
    return {"rel": 1e-5}


# ---------------------------------------------------------------- the inputs

def _generator(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + part * 7919 + 17) & ((1 << 62) - 1))
    return g


def _values(c, shape, g, scale=None):
    """fp32 values of the case's distribution: N(0,1), Student-t(4) of unit
    variance, or N(0,1) with two channels twenty times larger; a row of
    ``scale`` multiplies each context."""
    x = torch.randn(shape, generator=g, device="cuda")
    if c["values"] == "student":
        s = torch.zeros(shape, device="cuda")
        for _ in range(4):
            s += torch.randn(shape, generator=g, device="cuda") ** 2
        x = x / torch.sqrt(s / 4) / math.sqrt(2.0)
        del s
    elif c["values"] == "outliers":
        x[..., 3] *= 20.0
        x[..., 17] *= 20.0
    if scale is not None:
        x *= scale
    if c["kind"] == "session" and c["dtype"] == "float16":
        x = x.to(torch.float16)
    return x


def _scales(c, seed):
    """Per context log-normal(0, 0.5) scales of K and V, [contexts, 1, 1]."""
    n = c["sequences"] * c["layers"] * c["heads"]
    if c["sequences"] == 1 or c["values"] != "normal":
        return torch.ones(n, 1, 1, device="cuda")
    return torch.exp(0.5 * torch.randn(n, 1, 1, generator=_generator(seed, 1), device="cuda"))


def _groups(c, per_token):
    """(first sequence, sequences, tokens) of runs of equal length that make at
    most CHUNK values each; tokens as ``per_token(length)`` gives them."""
    each = c["layers"] * c["heads"]
    out, first, lengths = [], 0, _lengths(c)
    while first < c["sequences"]:
        n, count = per_token(lengths[first]), 1
        while (first + count < c["sequences"] and per_token(lengths[first + count]) == n
               and (count + 1) * each * n * c["dim"] <= CHUNK):
            count += 1
        out.append((first, count, n))
        first += count
    return out


def _cached(c, seed):
    """The tokens in the caches before the call: (first context, K, V) with K and
    V [contexts][tokens][dim], group by group."""
    each = c["layers"] * c["heads"]
    scales = _scales(c, seed)
    for i, (first, count, n) in enumerate(_groups(c, lambda length: length)):
        if n:
            lo, m = first * each, count * each
            g = _generator(seed, 100 + i)
            sc = scales[lo:lo + m]
            yield lo, _values(c, (m, n, c["dim"]), g, sc), _values(c, (m, n, c["dim"]), g, sc)


def _fresh(c, seed):
    """The call's own inputs: new K and V [contexts][append][dim] and queries
    [queries][contexts][dim]."""
    n, d = c["sequences"] * c["layers"] * c["heads"], c["dim"]
    g, sc = _generator(seed, 2), _scales(c, seed)
    k = _values(c, (n, c["append"], d), g, sc) if c["append"] else None
    v = _values(c, (n, c["append"], d), g, sc) if c["append"] else None
    return k, v, _values(c, (c["queries"], n, d), g)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


class Caches:
    """The MHAs of a case, one a sequence and layer, and a plan over their heads."""

    def __init__(self, c):
        from adaptq_amd import _lib
        self.L, self.last_error = _lib.lib, _lib.last_error
        self.mhas, self.plans = [], []
        self.heads = c["heads"]
        for unit in range(c["sequences"] * c["layers"]):
            m = self.L.adaptq_mha_create(self.heads, c["dim"], _bits_of(c, unit % c["layers"]),
                                         c["v_bits"], c["capacity"], 42 ^ unit, c["v_mass"],
                                         c["hybrid"])
            if not m:
                raise RuntimeError(self.last_error())
            self.mhas.append(m)

    def plan(self, first, count):
        """A plan over the heads of ``count`` MHAs from ``first`` on."""
        ctx = [self.L.adaptq_mha_head(m, h) for m in self.mhas[first:first + count]
               for h in range(self.heads)]
        p = self.L.adaptq_plan_create((C.c_void_p * len(ctx))(*ctx), len(ctx))
        if not p:
            raise RuntimeError(self.last_error())
        self.plans.append(p)
        return p

    def __del__(self):
        torch.cuda.synchronize()
        for p in self.plans:
            self.L.adaptq_plan_destroy(p)
        for m in self.mhas:
            self.L.adaptq_mha_destroy(m)


def prepare(c, seed):
    s = {"case": c, "stream": C.c_void_p(torch.cuda.current_stream().cuda_stream)}
    k, v, q = _fresh(c, seed)
    heads, layers, dim = c["heads"], c["layers"], c["dim"]
    if c["kind"] == "session":
        from adaptq_amd import AdaptQAttention
        s["module"] = AdaptQAttention(dim, heads, c["k_bits"], c["v_bits"], c["capacity"])
        qs = _values(c, (c["append"], 1, heads, dim), _generator(seed, 3))
        s["steps"] = [(qs[t], k[None, :, t].contiguous(), v[None, :, t].contiguous())
                      for t in range(c["append"])]
        return s
    if c["kind"] == "engine":
        from adaptq_amd import Engine
        e = Engine(dim, heads, c["k_bits"], c["v_bits"], c["capacity"], 42, c["v_mass"],
                   c["hybrid"])
        for _, ck, cv in _cached(c, seed):
            ck, cv = (x.transpose(0, 1).contiguous().cpu().numpy() for x in (ck, cv))
            for t in range(len(ck)):
                e.append(ck[t], cv[t])
        s.update(engine=e, k=k[:, 0].cpu().numpy(), v=v[:, 0].cpu().numpy(), q=q[0].cpu().numpy())
        return s
    s["caches"] = caches = Caches(c)
    L = caches.L
    for lo, ck, cv in _cached(c, seed):
        n = ck.shape[1]
        if c["first_k_bits"]:  # layers of other bits are no one plan
            for i in range(0, ck.shape[0], heads):
                m = caches.mhas[(lo + i) // heads]
                if L.adaptq_mha_append_all_device(m, _ptr(ck[i:]), _ptr(cv[i:]), n, 0,
                                                  s["stream"]):
                    raise RuntimeError(caches.last_error())
        elif L.adaptq_plan_append_device(caches.plan(lo // heads, ck.shape[0] // heads), _ptr(ck),
                                         _ptr(cv), n, 0, s["stream"]):
            raise RuntimeError(caches.last_error())
        torch.cuda.synchronize()
        del ck, cv
    out = torch.empty_like(q)
    s.update(k=k, v=v, q=q, out=out)
    if c["kind"] == "layers":
        s["calls"] = [(m, _ptr(k[i * heads:]), _ptr(v[i * heads:]), _ptr(q[0, i * heads:]),
                       _ptr(out[0, i * heads:])) for i, m in enumerate(caches.mhas)]
    elif c["kind"] in ("plan", "prefill"):
        s["plan"] = caches.plan(0, c["sequences"] * layers)
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "session":
        module = s["module"]
        module.reset_cache()
        return [torch.cat([module(q, k, v) for q, k, v in s["steps"]])]
    if c["kind"] == "engine":
        s["engine"].append(s["k"], s["v"])
        return [s["engine"].compute(s["q"])]
    caches, stream, out = s["caches"], s["stream"], s["out"]
    L, bad = caches.L, 0
    if c["kind"] == "layers":
        for m, k, v, q, o in s["calls"]:
            bad |= L.adaptq_mha_append_compute_all_device(m, k, v, c["tokens"], q, o, stream) < 0
    elif c["kind"] == "queries":
        row = 4 * c["dim"]
        bad = L.adaptq_ggml_attn_f32_device(caches.mhas[0], _ptr(s["q"]), c["dim"], c["heads"],
                                            c["queries"], row, c["heads"] * row, _ptr(out), row,
                                            c["heads"] * row, stream) < 0
    else:
        if c["append"]:
            bad |= L.adaptq_plan_append_device(s["plan"], _ptr(s["k"]), _ptr(s["v"]), c["append"],
                                               c["tokens"], stream) != 0
        bad |= L.adaptq_plan_compute_device(s["plan"], _ptr(s["q"]), _ptr(out), stream) != 0
    if bad:
        raise RuntimeError(caches.last_error())
    return [out]


# ------------------------------------------------------- the answer in 64 bits

def _signs(c, first, count):
    """The +-1 signs of ``count`` contexts from ``first`` on, [padded][count]:
    xorshift64 from the head's seed, odd states +1."""
    p, heads = _padded(c["dim"]), c["heads"]
    one = c["kind"] in ("session", "engine")
    seed = np.array([(42 if one else 42 ^ (i // heads)) ^ ((i % heads) * 0xDEADBEEFCAFE & U64)
                     for i in range(first, first + count)], np.uint64)
    out = np.empty((p, count), np.float32)
    s = np.where(seed == 0, np.uint64(0xDEADBEEFCAFE1234), seed)
    for i in range(p):
        s = s ^ (s << np.uint64(13))
        s = s ^ (s >> np.uint64(7))
        s = s ^ (s << np.uint64(17))
        out[i] = np.where(s & np.uint64(1), 1.0, -1.0)
    return torch.from_numpy(out).cuda()


def _butterflies(x):
    """The Hadamard transform over the first dimension, stage by stage, each sum
    rounded to x's own type."""
    p, size = x.shape[0], 1
    rest = x.shape[1:]
    while size < p:
        y = x.reshape(p // (2 * size), 2, size, *rest)
        x = torch.stack((y[:, 0] + y[:, 1], y[:, 0] - y[:, 1]), 1).reshape(p, *rest)
        size *= 2
    return x


def _coded(x, signs, bits):
    """Rows x [contexts][tokens][dim] as the cache holds them: (values [padded]
    [contexts][tokens] in 64 bits, scales in 64 bits).  Norms, rotation and codes
    in 32 bits, which is what defines the codes; the reference's clamp at three
    standard deviations lies above every threshold and changes none."""
    p = signs.shape[0]
    t = x.permute(2, 0, 1).contiguous()
    if t.shape[0] < p:
        t = torch.cat((t, torch.zeros(p - t.shape[0], *t.shape[1:], device=t.device)))
    if bits == 16:
        return t.double(), torch.ones(t.shape[1:], dtype=torch.float64, device=t.device)
    total = torch.zeros_like(t[0])
    for i in range(x.shape[2]):
        total = total + t[i] * t[i]
    norm = (total + np.float32(1e-12)).double().sqrt().float()
    t = t * norm.double().reciprocal().float() * signs[:, :, None]
    t = _butterflies(t)
    root = np.float32(np.sqrt(np.float64(p)))
    t = t * float(np.float32(1.0) / root) * float(root)
    book = np.array(CODEBOOK[bits], np.float32)
    codes = torch.zeros(t.shape, dtype=torch.uint8, device=t.device)
    for i in range(len(book) - 1):
        mid = np.float32(0) if i == len(book) // 2 - 1 else (book[i] + book[i + 1]) * np.float32(.5)
        codes += t >= float(mid)
    return torch.from_numpy(book.astype(np.float64)).cuda()[codes.int()], norm.double()


def _selected(w, mass):
    """Weights w [contexts][tokens] with those outside the heaviest ``mass`` of
    them left out: whole fours in descending order while the mass is short of it,
    then single tokens."""
    s, order = torch.sort(w, dim=1, descending=True, stable=True)
    n = w.shape[1]
    before = torch.cumsum(s, 1) - s
    i = torch.arange(n, device=w.device)
    start = torch.where(i // 4 * 4 + 3 < n, i // 4 * 4, i)
    s = torch.where(before[:, start] < float(np.float32(mass)), s, torch.zeros_like(s))
    return torch.zeros_like(w).scatter(1, order, s)


def _attend(c, k, v, q, signs, k_bits, mirror):
    """Attention of q [queries][contexts][dim] over rows k, v [contexts][tokens]
    [dim], [queries][contexts][dim] in 64 bits."""
    p, dim = signs.shape
    dim = c["dim"]
    v_bits = 16 if mirror else c["v_bits"]
    k_bits = 16 if mirror else k_bits
    sg = signs.double()
    kd, ks = _coded(k, signs, k_bits)
    weights = []
    for one in q.double():
        r = torch.zeros(p, one.shape[0], dtype=torch.float64, device=one.device)
        r[:dim] = one.t()
        if k_bits != 16:
            r = _butterflies(r * sg) / p
        logits = (kd * r[:, :, None]).sum(0) * ks / math.sqrt(dim)
        w = torch.softmax(logits, 1)
        if c["v_mass"] > 0 and k_bits != 16:
            w = _selected(w, c["v_mass"])
        weights.append(w)
    del kd
    vd, vs = _coded(v, signs, v_bits)
    outs = []
    for w in weights:
        acc = (vd * (w * vs)).sum(2)
        if v_bits != 16:
            acc = _butterflies(acc) * sg / p
        outs.append(acc[:dim].t())
    return torch.stack(outs)


def exact(c, seed):
    heads, each = c["heads"], c["layers"] * c["heads"]
    k, v, q = _fresh(c, seed)
    if c["kind"] == "session":  # token t over tokens 0..t, unquantised
        qs = _values(c, (c["append"], 1, heads, c["dim"]), _generator(seed, 3))[:, 0].double()
        kd, vd = k.double(), v.double()
        outs = []
        for t in range(c["append"]):
            w = (kd[:, :t + 1] * qs[t][:, None]).sum(2) / math.sqrt(c["dim"])
            outs.append((torch.softmax(w, 1)[:, :, None] * vd[:, :t + 1]).sum(1))
        return [torch.stack(outs)]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    blocks = _cached(c, seed) if c["tokens"] else [(0, None, None)]
    for lo, ck, cv in blocks:
        count = ck.shape[0] if ck is not None else k.shape[0]
        n = (ck.shape[1] if ck is not None else 0) + c["append"]
        mirror = c["hybrid"] >= n and n <= c["capacity"]
        step = heads
        while step * 2 <= each and each % (step * 2) == 0 and not c["first_k_bits"] \
                and step * 2 * n * _padded(c["dim"]) <= 1 << 28:
            step *= 2
        for i in range(0, count, step):
            at = slice(lo + i, lo + i + step)
            rows = []
            for old, new in ((ck, k), (cv, v)):
                parts = [x for x in (old[i:i + step] if old is not None else None,
                                     new[at] if new is not None else None) if x is not None]
                rows.append((torch.cat(parts, 1) if len(parts) > 1 else parts[0])
                            [:, -c["capacity"]:])
            bits = _bits_of(c, (lo + i) // heads % c["layers"])
            out[:, at] = _attend(c, rows[0], rows[1], q[:, at], _signs(c, lo + i, step), bits,
                                 mirror)
        del ck, cv
    return [out]
