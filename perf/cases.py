"""What this library is timed on: the calls of a paged-KV inference program, through HipExecutor.

Every case is one pass of such a program (one synchronous call, or one forward pass from
beginForwardPassCB to flushForwardPassCB), on buffers, weights and page tables that the program
already has on the device.  Kinds:

  decode   paged decode attention, one query row per request; with "write" the pass first puts
           every request's new K and V row into its page, as each layer of a decode step does
  prefill  chunked prefill attention over the paged cache
  model    decoder layers around the attention (and the output matrix), encoded call by call or
           replayed from a captured pass
  linear   one quantised projection over the rows of a prompt chunk or a batch
  kv_copy  a prompt's K and V rows written to pages and read back as contiguous rows
"""
from __future__ import annotations

import numpy as np
import torch

from mlcompiler_amd import HipExecutor
from mlcompiler_amd.workloads import q4_0_row_bytes, q6_k_row_bytes, rotary_tables

# hidden, query heads, KV heads, head_dim, FFN width, vocabulary of the two model shapes that the
# benchmark and the tests use
SHAPES = {"1b": (2048, 32, 4, 64, 5632, 32000), "8b": (4096, 32, 8, 128, 14336, 32000)}


def listed():
    return [
        # one user, one call per token: nothing but latency
        dict(name="decode_single", kind="decode", batch=1, heads=32, kv_heads=4, head_dim=64, page=64,
             ctx_lo=512, ctx_hi=512, ctx_seed=1, outliers=0.0, write=False),
        # the benchmark's headline: a served batch of mixed contexts
        dict(name="decode_b32", kind="decode", batch=32, heads=32, kv_heads=4, head_dim=64, page=64,
             ctx_lo=128, ctx_hi=2048, ctx_seed=2, outliers=0.0, write=False),
        # the attention part of a layer in a decode step: new K row, new V row, attention
        dict(name="decode_write_b64", kind="decode", batch=64, heads=32, kv_heads=4, head_dim=64, page=64,
             ctx_lo=256, ctx_hi=4096, ctx_seed=3, outliers=0.0, write=True),
        # long contexts, large heads, some keys far larger than the rest (softmax maxima move)
        dict(name="decode_long_b64", kind="decode", batch=64, heads=32, kv_heads=8, head_dim=128, page=64,
             ctx_lo=1024, ctx_hi=8192, ctx_seed=4, outliers=0.01, write=False),
        # three query heads per KV head and a cache of small pages
        dict(name="decode_ratio3_small_pages", kind="decode", batch=12, heads=24, kv_heads=8, head_dim=128, page=16,
             ctx_lo=100, ctx_hi=3000, ctx_seed=5, outliers=0.0, write=False),
        # the benchmark's chunked prefill: a 256-token chunk behind 3840 cached tokens
        dict(name="prefill_chunk_b8", kind="prefill", batch=8, chunk=256, heads=32, kv_heads=8, head_dim=128, page=64,
             ctx_lo=3840, ctx_hi=3840, ctx_seed=6),
        # short prompts that arrive together, no size a multiple of anything
        dict(name="prefill_ragged_b3", kind="prefill", batch=3, chunk=77, heads=32, kv_heads=4, head_dim=64, page=64,
             ctx_lo=0, ctx_hi=900, ctx_seed=7),
        # one layer of the larger shape as the batched walker drives it, operator by operator
        dict(name="layer_8b_b16", kind="model", shape="8b", layers=1, head=False, replay=False, batch=16,
             ctx_lo=512, ctx_hi=4096, ctx_seed=8),
        # whole decode steps, replayed from a captured pass: one user, and a served batch
        dict(name="step_1b_b1", kind="model", shape="1b", layers=22, head=True, replay=True, batch=1,
             ctx_lo=600, ctx_hi=600, ctx_seed=9),
        dict(name="step_1b_b32", kind="model", shape="1b", layers=22, head=True, replay=True, batch=32,
             ctx_lo=128, ctx_hi=2048, ctx_seed=2),
        # a projection over the rows of a prompt chunk
        dict(name="linear_q4_chunk512", kind="linear", format="q4_0", rows=11264, cols=2048, tokens=512),
        # a prompt's rows moved into the paged cache and out again
        dict(name="kv_copy_1500", kind="kv_copy", tokens=1500, kv_heads=8, head_dim=128, page=64, start=0, dtype_bytes=2),
    ]


def _log(rng, lo, hi):
    """A whole number, spread over the logarithm of [lo, hi]."""
    return int(min(hi, max(lo, round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case of the same ranges.  Batches shrink until the case costs no more than the
    largest listed ones (1.2 GB of cache read, 130 GFLOP)."""
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "model", "linear", "linear", "kv_copy"])
    seed = rng.randrange(1 << 20)
    if kind == "decode":
        kv, ratio, d = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 3, 4, 4, 6, 8, 8, 16]), rng.choice([64, 128])
        hi = _log(rng, 16, 8192)
        most = int(1.1e9 / (hi * 4 * kv * d))
        return dict(kind="decode", batch=_log(rng, 1, max(1, min(128, most))), heads=kv * ratio, kv_heads=kv, head_dim=d,
                    page=rng.choice([16, 32, 64, 64, 64, 128]), ctx_lo=max(1, hi // rng.choice([1, 4, 16])), ctx_hi=hi,
                    ctx_seed=seed, outliers=rng.choice([0.0, 0.0, 0.01]), write=rng.random() < 0.4)
    if kind == "prefill":
        kv, ratio, d = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 4, 8, 8]), rng.choice([64, 128])
        chunk, hi = _log(rng, 16, 1024), rng.choice([0, _log(rng, 16, 8192)])
        most = int(1.3e11 / (4.0 * d * kv * ratio * chunk * (hi + chunk)))
        return dict(kind="prefill", batch=_log(rng, 1, max(1, min(8, most))), chunk=chunk, heads=kv * ratio, kv_heads=kv,
                    head_dim=d, page=rng.choice([32, 64, 64, 128]), ctx_lo=hi // rng.choice([1, 4]), ctx_hi=hi, ctx_seed=seed)
    if kind == "model":
        shape = rng.choice(["1b", "1b", "8b"])
        hi, replay = _log(rng, 64, 4096), rng.random() < 0.7
        most = 64 if shape == "1b" else int(1.1e9 / (hi * 4096 * 2))
        layers = _log(rng, 1, 22) if shape == "1b" else rng.choice([1, 2])
        return dict(kind="model", shape=shape, layers=layers, head=shape == "1b" and rng.random() < 0.5, replay=replay,
                    batch=_log(rng, 1, max(1, min(64, most))), ctx_lo=max(1, hi // 4), ctx_hi=hi, ctx_seed=seed)
    if kind == "linear":
        fmt = rng.choice(["q4_0", "q4_0", "q6_k"])
        rows, cols = rng.choice([(2560, 2048), (2048, 2048), (11264, 2048), (2048, 5632), (6144, 4096), (4096, 4096),
                                 (28672, 4096), (4096, 14336)] if fmt == "q4_0" else [(32000, 2048), (2048, 2048), (4096, 4096)])
        return dict(kind="linear", format=fmt, rows=rows, cols=cols,
                    tokens=_log(rng, 1, max(1, min(2048, int(1.0e11 / (2.0 * rows * cols))))))
    page = rng.choice([16, 64, 64, 128])
    return dict(kind="kv_copy", tokens=_log(rng, 1, 8192), kv_heads=rng.choice([2, 4, 8]), head_dim=rng.choice([64, 128]),
                page=page, start=rng.choice([0, rng.randrange(page)]), dtype_bytes=rng.choice([2, 2, 4]))


# ---- sizes that follow from a case ----------------------------------------------------------

def _contexts(c):
    """Context lengths (decode: the new token included; prefill: cached tokens), the case's own."""
    return np.random.default_rng(c["ctx_seed"]).integers(c["ctx_lo"], c["ctx_hi"] + 1, c["batch"]).astype(np.int64)


def _projections(shape):
    hidden, heads, kv, d, ffn, _ = SHAPES[shape]
    return dict(qkv=((heads + 2 * kv) * d, hidden), o=(hidden, heads * d), gate_up=(2 * ffn, hidden), down=(hidden, ffn))


def work(c):
    if c["kind"] == "decode":
        n = int(_contexts(c).sum())
        io = 8 * c["batch"] * c["heads"] * c["head_dim"] + (8 * c["batch"] * c["kv_heads"] * c["head_dim"] if c["write"] else 0)
        return {"bytes": n * 4 * c["kv_heads"] * c["head_dim"] + io, "flops": 4 * n * c["heads"] * c["head_dim"]}
    if c["kind"] == "prefill":
        ctx, m = _contexts(c), c["chunk"]
        seen = int((ctx * m + m * (m + 1) // 2).sum())
        kv = int((ctx + m).sum()) * 4 * c["kv_heads"] * c["head_dim"]
        return {"bytes": kv + 6 * c["batch"] * m * c["heads"] * c["head_dim"], "flops": 4 * seen * c["heads"] * c["head_dim"]}
    if c["kind"] == "model":
        hidden, heads, kv, d, _, vocab = SHAPES[c["shape"]]
        n, b, mats = int(_contexts(c).sum()), c["batch"], _projections(c["shape"]).values()
        layer = sum(r * q4_0_row_bytes(k) for r, k in mats) + n * 4 * kv * d + 8 * b * hidden
        flops = sum(2 * r * k * b for r, k in mats) + 4 * n * heads * d
        out = vocab * q6_k_row_bytes(hidden) + 4 * b * (vocab + hidden) if c["head"] else 0
        return {"bytes": c["layers"] * layer + out, "flops": c["layers"] * flops + (2 * vocab * hidden * b if c["head"] else 0)}
    if c["kind"] == "linear":
        row = q4_0_row_bytes(c["cols"]) if c["format"] == "q4_0" else q6_k_row_bytes(c["cols"])
        return {"bytes": c["rows"] * row + 4 * c["tokens"] * (c["rows"] + c["cols"]), "flops": 2 * c["rows"] * c["cols"] * c["tokens"]}
    row = c["kv_heads"] * c["head_dim"] * c["dtype_bytes"]
    return {"bytes": 2 * row * (2 * c["tokens"] + 2 * (c["tokens"] + c["start"])), "flops": 0}


def tolerance(c):
    if c["kind"] == "decode":   # fp16 cache, everything else fp32; large scores magnify the rounding of their sums
        return {"rel": 1e-4 if c["outliers"] else 2e-5}
    if c["kind"] == "prefill":  # softmax weights enter the second product as fp16
        return {"rel": 1e-3}
    if c["kind"] == "model":    # fp32 sums through the layers; a K or V element may round to the next fp16 number
        return {"rel": 2e-4, "max": 2e-2}
    if c["kind"] == "linear":
        return {"rel": 1e-5}
    return "exact"


# ---- inputs ---------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator("cuda").manual_seed(seed)


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _tables(seed, lengths, page, spare=3):
    """Page tables over a shuffled pool: flat ids, offsets, pages of the pool."""
    pages = (lengths + page - 1) // page
    off = np.zeros(len(lengths) + 1, np.uint32)
    off[1:] = np.cumsum(pages)
    pool = int(pages.sum()) + spare
    flat = np.random.default_rng(seed).permutation(pool).astype(np.uint32)[:int(pages.sum())]
    return flat, off, pool


def _q4_matrix(g, rows, cols):
    """Q4_0 rows of weights that are spread like a normal variable (deviation 0.03 and less)."""
    nb = cols // 32
    codes = (_normal(g, rows, nb, 32) * 2.7 + 8.0).round().clamp(0, 15).to(torch.uint8)
    d = (0.008 + 0.003 * torch.rand(rows, nb, 1, generator=g, device="cuda")).half()
    return torch.cat([d.view(torch.uint8), codes[..., :16] | (codes[..., 16:] << 4)], 2).reshape(rows, nb * 18).cpu().numpy()


def _q6_matrix(g, rows, cols):
    nb = cols // 256
    codes = torch.randint(0, 256, (rows, nb, 192), generator=g, device="cuda", dtype=torch.uint8)
    scales = torch.randint(32, 128, (rows, nb, 16), generator=g, device="cuda", dtype=torch.uint8)
    d = (1.6e-5 + 6e-6 * torch.rand(rows, nb, 1, generator=g, device="cuda")).half()
    return torch.cat([codes, scales, d.view(torch.uint8)], 2).reshape(rows, nb * 210).cpu().numpy()


def _ok(exe, done):
    if not done:
        raise RuntimeError(exe.lastError())


class _Decode:
    def __init__(self, c, seed):
        self.exe, g = HipExecutor.Instance(), _gen(seed)
        b, h, kv, d, p = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["page"]
        n = _contexts(c)
        self.flat, self.off, pool = _tables(seed, n, p)
        self.seq, self.pos = n.astype(np.uint32), (n - 1).astype(np.uint32)
        self.q, self.o = _normal(g, b, h, d), torch.zeros(b, h, d, device="cuda")
        self.k, self.v = (_normal(g, pool, p, kv, d, dtype=torch.float16) for _ in range(2))
        if c["outliers"]:
            self.k *= torch.where(torch.rand(pool, p, 1, 1, generator=g, device="cuda") < c["outliers"], 8.0, 1.0).half()
        self.new = _normal(g, 2, b, kv, d, dtype=torch.float16) if c["write"] else None
        self.ids, self.slots = self.flat[self.off[1:] - 1], self.pos % p
        self.rows = (p, kv, d, b)
        self.args = (self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(), self.o.data_ptr(), self.flat, self.off,
                     self.seq, self.pos, b, h, kv, d, p, True)

    def run(self):
        exe = self.exe
        if self.new is None:
            _ok(exe, exe.runPagedFlashAttention(*self.args))
            return self.o
        _ok(exe, exe.beginForwardPassCB())
        for pool, rows in ((self.k, self.new[0]), (self.v, self.new[1])):
            _ok(exe, exe.encodeScatterKVPagedBatched(pool.data_ptr(), self.ids, self.slots, *self.rows, rows.data_ptr()))
        _ok(exe, exe.encodePagedFlashAttention(*self.args))
        _ok(exe, exe.flushForwardPassCB())
        return self.o, self.k, self.v


class _Prefill:
    def __init__(self, c, seed):
        self.exe, g = HipExecutor.Instance(), _gen(seed)
        b, m, h, kv, d, p = c["batch"], c["chunk"], c["heads"], c["kv_heads"], c["head_dim"], c["page"]
        cached = _contexts(c)
        flat, off, pool = _tables(seed, cached + m, p)
        self.q = _normal(g, b, m, h, d, dtype=torch.float16)
        self.k, self.v = (_normal(g, pool, p, kv, d, dtype=torch.float16) for _ in range(2))
        self.o = torch.zeros(b, m, h, d, device="cuda")
        self.args = (self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(), self.o.data_ptr(), flat, off,
                     (cached + m).astype(np.uint32), cached.astype(np.uint32), b, m, h, kv, d, p)

    def run(self):
        _ok(self.exe, self.exe.runPagedPrefillAttention(*self.args))
        return self.o


class _Model:
    """Decoder layers as the batched walker drives them; all layers have the same weights' values,
    each its own copy on the device."""

    def __init__(self, c, seed):
        self.exe, g = HipExecutor.Instance(), _gen(seed)
        self.c, b = c, c["batch"]
        hidden, h, kv, d, ffn, vocab = SHAPES[c["shape"]]
        n = _contexts(c)
        self.flat, self.off, pool = _tables(seed, n, 64)
        self.seq, self.pos = n.astype(np.uint32), (n - 1).astype(np.uint32)
        self.ids, self.slots = self.flat[self.off[1:] - 1], self.pos % 64
        self.names = "%s.%d" % (c["shape"], seed)
        self.mats = {m: _q4_matrix(g, *s) for m, s in _projections(c["shape"]).items()}
        self.mats["head"] = _q6_matrix(g, vocab, hidden) if c["head"] else None
        rng = np.random.default_rng(seed)
        self.norms = [rng.uniform(0.5, 1.5, hidden).astype(np.float32) for _ in range(2 * c["layers"] + 1)]
        self.x = _normal(g, b, hidden)
        self.pools = _normal(g, c["layers"], 2, pool, 64, kv, d, dtype=torch.float16)
        self.rows16 = torch.zeros(c["layers"], 2, b, kv * d, device="cuda", dtype=torch.float16)
        self.rotary = [torch.from_numpy(t).cuda() for t in rotary_tables(self.pos, d)]
        f = dict(norm=hidden, qkv=(h + 2 * kv) * d, q=h * d, k=kv * d, v=kv * d, attn=h * d, o=hidden, resid=hidden,
                 gate_up=2 * ffn, gate=ffn, up=ffn, mix=ffn, down=hidden, out0=hidden, out1=hidden,
                 logits=vocab if c["head"] else 1)
        self.f = {name: torch.zeros(b, width, device="cuda") for name, width in f.items()}
        torch.cuda.synchronize()
        self.handle = 0
        self.call_by_call()          # brings weights and tables to the device
        if c["replay"]:
            self.capture()

    def encode(self):
        exe, c, b = self.exe, self.c, self.c["batch"]
        hidden, h, kv, d, ffn, vocab = SHAPES[c["shape"]]
        p = {name: t.data_ptr() for name, t in self.f.items()}
        cos, sin = (t.data_ptr() for t in self.rotary)
        proj = _projections(c["shape"])

        def matmul(m, layer, src, dst):
            rows, cols = proj[m]
            w = self.mats[m]
            _ok(exe, exe.encodeMatMulQ4_0Batched("%s.%d.%s" % (self.names, layer, m), w, p[src] if src in p else src, b, rows,
                                                 cols, w.shape[1], 2, p[dst]))

        x = self.x.data_ptr()
        for i in range(c["layers"]):
            out = p["out%d" % (i % 2)]
            pages, row16 = ([t.data_ptr() for t in s[i]] for s in (self.pools, self.rows16))
            _ok(exe, exe.encodeRmsNormBatched(x, self.norms[2 * i], 1e-5, b, hidden, p["norm"]))
            matmul("qkv", i, "norm", "qkv")
            _ok(exe, exe.encodeQkvSplitRopeCast(p["qkv"], p["q"], p["k"], p["v"], *row16, cos, sin, b, h, kv, d,
                                                (h + 2 * kv) * d, h * d, kv * d, kv * d, d))
            for pool, rows in zip(pages, row16):
                _ok(exe, exe.encodeScatterKVPagedBatched(pool, self.ids, self.slots, 64, kv, d, b, rows))
            _ok(exe, exe.encodePagedFlashAttention(p["q"], *pages, p["attn"], self.flat, self.off, self.seq, self.pos, b, h, kv,
                                                   d, 64, True))
            matmul("o", i, "attn", "o")
            _ok(exe, exe.encodeAddBatched(p["o"], x, p["resid"], b * hidden))
            _ok(exe, exe.encodeRmsNormBatched(p["resid"], self.norms[2 * i + 1], 1e-5, b, hidden, p["norm"]))
            matmul("gate_up", i, "norm", "gate_up")
            _ok(exe, exe.encodeGateUpSplitSiluMul(p["gate_up"], p["gate"], p["up"], p["mix"], b, ffn, 2 * ffn))
            matmul("down", i, "mix", "down")
            _ok(exe, exe.encodeAddBatched(p["down"], p["resid"], out, b * hidden))
            x = out
        if c["head"]:
            w = self.mats["head"]
            _ok(exe, exe.encodeRmsNormBatched(x, self.norms[-1], 1e-5, b, hidden, p["norm"]))
            _ok(exe, exe.encodeMatMulQ6KBatched("%s.head" % self.names, w, p["norm"], b, vocab, hidden, w.shape[1], p["logits"]))

    def call_by_call(self):
        _ok(self.exe, self.exe.beginForwardPassCB())
        self.encode()
        _ok(self.exe, self.exe.flushForwardPassCB())

    def capture(self):
        exe = self.exe
        if self.handle:              # the pass has to be recorded anew: bring everything up to date first
            exe.captureRelease(self.handle)
            self.call_by_call()
        _ok(exe, exe.beginForwardPassCB() and exe.captureBegin())
        self.encode()
        self.handle = exe.captureEnd()
        _ok(exe, self.handle > 0 and exe.flushForwardPassCB())

    def run(self):
        exe = self.exe
        if self.c["replay"]:
            step = (self.flat, self.off, self.seq, self.pos, self.ids, self.slots)
            if not exe.replayUpdate(self.handle, *step):
                self.capture()
                _ok(exe, exe.replayUpdate(self.handle, *step))
            _ok(exe, exe.beginForwardPassCB() and exe.replay(self.handle) and exe.flushForwardPassCB())
        else:
            self.call_by_call()
        out = self.f["logits"] if self.c["head"] else self.f["out%d" % ((self.c["layers"] - 1) % 2)]
        return out, self.rows16, self.pools

    def __del__(self):
        if getattr(self, "handle", 0):
            self.exe.captureRelease(self.handle)


class _Linear:
    def __init__(self, c, seed):
        self.exe, g = HipExecutor.Instance(), _gen(seed)
        q4, rows, cols, m = c["format"] == "q4_0", c["rows"], c["cols"], c["tokens"]
        self.w = (_q4_matrix if q4 else _q6_matrix)(g, rows, cols)
        self.x, self.out = _normal(g, m, cols), torch.zeros(m, rows, device="cuda")
        name = "linear.%s.%dx%d.%d" % (c["format"], rows, cols, seed)
        self.call = self.exe.encodeMatMulQ4_0Batched if q4 else self.exe.encodeMatMulQ6KBatched
        self.args = (name, self.w, self.x.data_ptr(), m, rows, cols, self.w.shape[1]) + ((2,) if q4 else ()) + (self.out.data_ptr(), True)
        torch.cuda.synchronize()
        self.run()                   # the weights reach the device with the first call that names them

    def run(self):
        _ok(self.exe, self.call(*self.args))
        return self.out


class _KvCopy:
    def __init__(self, c, seed):
        self.exe, g = HipExecutor.Instance(), _gen(seed)
        kv, d, p, n, start = c["kv_heads"], c["head_dim"], c["page"], c["tokens"], c["start"]
        t = torch.float16 if c["dtype_bytes"] == 2 else torch.float32
        self.table, _, pool = _tables(seed, np.array([n + start]), p)
        self.src = [_normal(g, kv, n, d, dtype=t) for _ in range(2)]
        self.pool = [_normal(g, pool, p, kv, d, dtype=t) for _ in range(2)]
        self.dst = [torch.zeros(kv, n + start, d, device="cuda", dtype=t) for _ in range(2)]
        self.c = c

    def run(self):
        exe, c = self.exe, self.c
        kv, d, p, n, start, size = (c[x] for x in ("kv_heads", "head_dim", "page", "tokens", "start", "dtype_bytes"))
        for src, pool in zip(self.src, self.pool):
            _ok(exe, exe.scatterKVPaged(pool.data_ptr(), self.table, p, kv, d, n, start, src.data_ptr(), size))
        for pool, dst in zip(self.pool, self.dst):
            _ok(exe, exe.gatherKVPages(pool.data_ptr(), self.table, p, kv, d, n + start, dst.data_ptr(), size))
        return self.dst + self.pool


def prepare(case, seed):
    HipExecutor.Instance().requireAvailable()
    kinds = {"decode": _Decode, "prefill": _Prefill, "model": _Model, "linear": _Linear, "kv_copy": _KvCopy}
    state = kinds[case["kind"]](case, seed)
    torch.cuda.synchronize()         # torch's stream and the library's are not ordered with each other
    return state


def run(state):
    return state.run()
