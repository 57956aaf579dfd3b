"""Q4_0 matmuls in a row that hand each other their input in the library's own buffers: one that still reads such a
buffer while its epilogue writes the next one's.  Every result is checked against the float64 product of the GPU's own
input, as in test_matmul_tokens_gpu.py."""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4
from oracle import paged_oracle as po
from test_matmul_norm_fusion_gpu import EPS, _pool, _read
from test_matmul_tokens_gpu import check

pytestmark = pytest.mark.gpu


def _weights(rng, rows, cols):
    return po.quantize_q4_0((rng.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float32))


@pytest.mark.parametrize("batch,widths,fused", [
    # as many workgroups as CUs in the middle: the first write the next input, which is wider than their own, when
    # others still read theirs
    (64, (64, 2048, 4096, 8192), 2),
    (33, (160, 3072, 4096, 8192), 2),               # four tiles each, of 16 waves and at the end of 8
    (21, (160, 4096, 10240), 1), (32, (160, 2048, 10240), 1),   # the reader's workgroups have two groups of requests each
    (16, (128, 512, 512, 1024, 512, 1024), 4),      # the buffers change three times
    (5, (64, 1024, 256, 4096), 2),                  # ... get narrower, and wider
])
def test_norms_in_a_row(exe, batch, widths, fused):
    """matmul, add, norm, matmul, add, norm, ... matmul"""
    rng = np.random.default_rng(batch)
    n = len(widths) - 1
    w = [_weights(rng, widths[i + 1], widths[i]) for i in range(n)]
    x = rng.standard_normal((batch, widths[0])).astype(np.float32)
    resid = [rng.standard_normal((batch, v)).astype(np.float32) for v in widths[1:-1]]
    gamma = [(1.0 + 0.3 * rng.standard_normal(v)).astype(np.float32) for v in widths[1:-1]]
    like = {f"{m}{i}": np.empty((batch, widths[i + 1]), np.float32) for i in range(n) for m in "phn"}
    dev = {m: _pool(exe, np.full_like(a, np.nan)) for m, a in like.items()}
    src = [_pool(exe, a) for a in [x] + resid]
    before = exe.fusedMatmulNormLaunches()
    try:
        for _ in range(2):       # (the second pass finds its buffers as the first left them)
            a = src[0]
            assert exe.beginForwardPassCB()
            for i in range(n):
                assert exe.encodeMatMulQ4_0Batched(f"row{batch}.{i}", w[i], a, batch, widths[i + 1], widths[i], w[i].shape[1], 1,
                                                   dev[f"p{i}"]), exe.lastError()
                if i < n - 1:
                    assert exe.encodeAddBatched(dev[f"p{i}"], src[i + 1], dev[f"h{i}"], batch * widths[i + 1])
                    assert exe.encodeRmsNormBatched(dev[f"h{i}"], gamma[i], EPS, batch, widths[i + 1], dev[f"n{i}"])
                    a = dev[f"n{i}"]
            assert exe.flushForwardPassCB(), exe.lastError()
            got = {m: _read(exe, dev[m], like[m]) for m in like}
            a = x
            for i in range(n):
                check(got[f"p{i}"], q4.dequant(w[i], widths[i]), a)
                if i < n - 1:
                    a = got[f"n{i}"]
                    assert np.array_equal(got[f"h{i}"], resid[i] + got[f"p{i}"])
                    want = po.rms_norm_batched(got[f"h{i}"], gamma[i], EPS, batch, widths[i + 1])
                    assert (np.abs(a - want) <= 2e-6 * np.abs(want).max(axis=1, keepdims=True)).all()
    finally:
        for buf in list(dev.values()) + src:
            exe.releaseScratchBuffer(buf)
    assert exe.fusedMatmulNormLaunches() - before == 2 * fused


@pytest.mark.parametrize("batch,ffn", [(32, (4128, 8192)), (3, (4160, 4128))])
def test_gate_up_behind_gate_up(exe, batch, ffn):
    """gate/up, split + SiLU, gate/up over the products, split + SiLU, matmul"""
    rng = np.random.default_rng(batch)
    hid, rows = 64, 192
    shapes = ((2 * ffn[0], hid), (2 * ffn[1], ffn[0]), (rows, ffn[1]))
    w = [_weights(rng, *s) for s in shapes]
    x = rng.standard_normal((batch, hid)).astype(np.float32)
    like = {f"{m}{i}": np.empty((batch, v * ffn[i]), np.float32) for i in range(2) for m, v in (("y", 2), ("g", 1), ("u", 1), ("m", 1))}
    like["y2"] = np.empty((batch, rows), np.float32)
    dev = {m: _pool(exe, np.full_like(a, np.nan)) for m, a in like.items()}
    d_x = _pool(exe, x)
    before = exe.fusedMatmulSiluSplitLaunches()
    try:
        assert exe.beginForwardPassCB()
        a = d_x
        for i, (r, c) in enumerate(shapes):
            assert exe.encodeMatMulQ4_0Batched(f"gu{batch}.{i}", w[i], a, batch, r, c, w[i].shape[1], 1, dev[f"y{i}"]), exe.lastError()
            if i < 2:
                a = dev[f"m{i}"]
                assert exe.encodeGateUpSplitSiluMul(dev[f"y{i}"], dev[f"g{i}"], dev[f"u{i}"], a, batch, ffn[i], 2 * ffn[i])
        assert exe.flushForwardPassCB(), exe.lastError()
        got = {m: _read(exe, dev[m], like[m]) for m in like}
    finally:
        for buf in list(dev.values()) + [d_x]:
            exe.releaseScratchBuffer(buf)
    assert exe.fusedMatmulSiluSplitLaunches() - before == 2
    for i, a in enumerate((x, got["m0"], got["m1"])):
        check(got[f"y{i}"], q4.dequant(w[i], shapes[i][1]), a)
    for i in range(2):
        _, _, want = po.gate_up_split_silu_mul(got[f"y{i}"], batch, ffn[i], 2 * ffn[i])
        assert np.max(np.abs(got[f"m{i}"] - want) / (np.abs(want) + 1e-30)) < 5e-6


@pytest.mark.parametrize("what", ["fragments", "weights", "norm_weights"])
def test_a_held_back_matmul_keeps_what_it_reads(exe, what):
    """Calls behind a held-back matmul that replace what it reads: a matmul with a longer row than any before it
    ("q4_x_fragments" grows; it has too few rows to take the norm over), another matrix under the same name, other norm
    weights in the same host array."""
    batch = 64 if what == "fragments" else 16
    widths = {"fragments": (64, 8192, 64), "weights": (256, 512, 1024), "norm_weights": (256, 512, 512, 1024)}[what]
    rng = np.random.default_rng(7)
    n = len(widths) - 1
    w = [_weights(rng, widths[i + 1], widths[i]) for i in range(n)]
    x = rng.standard_normal((batch, widths[0])).astype(np.float32)
    resid = [rng.standard_normal((batch, v)).astype(np.float32) for v in widths[1:-1]]
    gammas = [(1.0 + 0.3 * rng.standard_normal(v)).astype(np.float32) for v in widths[1:-1]]
    gamma = gammas[0].copy()
    like = {f"{m}{i}": np.empty((batch, widths[i + 1]), np.float32) for i in range(n) for m in "phn"}
    dev = {m: _pool(exe, np.full_like(a, np.nan)) for m, a in like.items()}
    src = [_pool(exe, a) for a in [x] + resid]
    try:
        a = src[0]
        assert exe.beginForwardPassCB()
        for i in range(n):
            name = "kept" if what == "weights" else f"kept.{what}.{i}"
            assert exe.encodeMatMulQ4_0Batched(name, w[i], a, batch, widths[i + 1], widths[i], w[i].shape[1], 1,
                                               dev[f"p{i}"]), exe.lastError()
            if i < n - 1:
                gamma[:] = gammas[i]
                a = dev[f"n{i}"]
                assert exe.encodeAddBatched(dev[f"p{i}"], src[i + 1], dev[f"h{i}"], batch * widths[i + 1])
                assert exe.encodeRmsNormBatched(dev[f"h{i}"], gamma, EPS, batch, widths[i + 1], a)
        assert exe.flushForwardPassCB(), exe.lastError()
        got = {m: _read(exe, dev[m], like[m]) for m in like}
    finally:
        for buf in list(dev.values()) + src:
            exe.releaseScratchBuffer(buf)
    a = x
    for i in range(n):
        check(got[f"p{i}"], q4.dequant(w[i], widths[i]), a)
        if i < n - 1:
            a = got[f"n{i}"]
            want = po.rms_norm_batched(got[f"h{i}"], gammas[i], EPS, batch, widths[i + 1])
            assert (np.abs(a - want) <= 2e-6 * np.abs(want).max(axis=1, keepdims=True)).all()


# Buffers that a chain  p0 = W0 x; h0 = r0 + p0; n0 = norm(h0); p1 = W1 n0; h1 = r1 + p1; n1 = norm(h1); y = W2 n1
# may share, as long as nobody reads what was overwritten: {buffer: the one that it is}, and how many of the two norms
# the matmuls can still take over then.
SHARED = {
    "sums_over_residuals": ({"h0": "r0", "h1": "r1"}, 2),
    "sum_over_the_sum_before": ({"h1": "h0"}, 1),
    "sum_over_the_norm_before": ({"h1": "n0"}, 1),
    "norm_before_as_residual": ({"r1": "n0"}, 1),
    "sum_before_as_residual": ({"r1": "h0"}, 2),
    "residual_over_and_over": ({"h0": "r0", "r1": "r0", "h1": "r0"}, 1),
    "output_over_the_sum_before": ({"p1": "h0"}, 1),
    "output_over_its_input": ({"p1": "n0"}, 1),
    "output_added_to_itself": ({"r1": "p1"}, 1),
    "sum_over_the_output": ({"h0": "p0", "h1": "p1"}, 2),
    "norms_in_place": ({"n0": "h0", "n1": "h1"}, 2),
    "last_output_over_the_sum": ({"y": "h1"}, 1),
    "last_output_over_the_norm": ({"y": "n1"}, 1),
    "everything_in_two": ({"p0": "x", "h0": "x", "n0": "x", "p1": "r0", "h1": "r0", "n1": "r0", "r1": "x", "y": "x"}, 1),
}


@pytest.mark.parametrize("batch", [3, 32])
@pytest.mark.parametrize("shared", list(SHARED), ids=list(SHARED))
def test_shared_buffers(exe, shared, batch):
    """The chain with its launches fused gives what its calls one by one give, whichever buffers are the same.
    (Tolerance as in test_row_chain_fuzz_gpu.py: the fused norm's sum runs in another order.)"""
    same, fused = SHARED[shared]
    rng = np.random.default_rng(batch)
    n = 512
    w = [_weights(rng, n, n) for _ in range(3)]
    gamma = [(1.0 + 0.3 * rng.standard_normal(n)).astype(np.float32) for _ in range(2)]
    init = {m: rng.standard_normal((batch, n)).astype(np.float32) for m in ("x", "r0", "r1", "p0", "h0", "n0", "p1", "h1", "n1", "y")}
    out = {}
    for fuse in (0, 1):
        dev = {m: _pool(exe, a) for m, a in init.items()}
        at = lambda m: dev[same.get(m, m)]
        assert exe.setOption("fuse_row_ops", fuse)
        before = exe.fusedMatmulNormLaunches()
        try:
            a = "x"
            assert exe.beginForwardPassCB()
            for i, dst in enumerate(("p0", "p1", "y")):
                assert exe.encodeMatMulQ4_0Batched(f"shared{batch}.{i}", w[i], at(a), batch, n, n, w[i].shape[1], 1, at(dst)), exe.lastError()
                if i < 2:
                    a = f"n{i}"
                    assert exe.encodeAddBatched(at(f"r{i}"), at(dst), at(f"h{i}"), batch * n)
                    assert exe.encodeRmsNormBatched(at(f"h{i}"), gamma[i], EPS, batch, n, at(a))
            assert exe.flushForwardPassCB(), exe.lastError()
            out[fuse] = {m: _read(exe, b, init[m]) for m, b in dev.items()}
        finally:
            exe.setOption("fuse_row_ops", 1)
            for buf in dev.values():
                exe.releaseScratchBuffer(buf)
        assert exe.fusedMatmulNormLaunches() - before == (fused if fuse else 0)
    for m, want in out[0].items():
        assert np.isfinite(want).all() and np.abs(out[1][m] - want).max() <= 1e-4 * np.abs(want).max(), m


@pytest.mark.parametrize("batch,rows,ksplit", [(8, 1536, 6), (5, 1088, 8), (8, 1536, 1), (8, 1536, 0)])
@pytest.mark.parametrize("in_place", [False, True])
def test_norm_in_front_of_k_slices(exe, batch, rows, ksplit, in_place):
    """A norm whose reader splits its K: every element is written, and once.  (Slices would each finish the norm, and have
    fewer row groups than the other forms.)"""
    rng = np.random.default_rng(ksplit)
    n = 4096
    w = [_weights(rng, n, 512), _weights(rng, rows, n)]
    gamma = (1.0 + 0.3 * rng.standard_normal(n)).astype(np.float32)
    init = {"x": rng.standard_normal((batch, 512)), "r": rng.standard_normal((batch, n)), "p": np.zeros((batch, n)),
            "h": np.full((batch, n), np.nan), "n": np.full((batch, n), np.nan), "y": np.full((batch, rows), np.nan)}
    dev = {m: _pool(exe, a.astype(np.float32)) for m, a in init.items()}
    norm = dev["h" if in_place else "n"]
    before = exe.fusedMatmulNormLaunches()
    assert exe.setOption("q4_ksplit", ksplit)
    try:
        assert exe.beginForwardPassCB()
        assert exe.encodeMatMulQ4_0Batched(f"sliced.{ksplit}.0", w[0], dev["x"], batch, n, 512, w[0].shape[1], 1, dev["p"]), exe.lastError()
        assert exe.encodeAddBatched(dev["p"], dev["r"], dev["h"], batch * n)
        assert exe.encodeRmsNormBatched(dev["h"], gamma, EPS, batch, n, norm)
        assert exe.encodeMatMulQ4_0Batched(f"sliced.{ksplit}.{rows}", w[1], norm, batch, rows, n, w[1].shape[1], 1, dev["y"]), exe.lastError()
        assert exe.flushForwardPassCB(), exe.lastError()
        got = {m: _read(exe, b, np.empty(init[m].shape, np.float32)) for m, b in dev.items()}
    finally:
        exe.setOption("q4_ksplit", 0)
        for buf in dev.values():
            exe.releaseScratchBuffer(buf)
    total = got["r"] + got["p"]
    want = po.rms_norm_batched(total, gamma, EPS, batch, n)
    if not in_place:
        assert np.array_equal(got["h"], total)
    a = got["h" if in_place else "n"]
    assert (np.abs(a - want) <= 2e-6 * np.abs(want).max(axis=1, keepdims=True)).all()
    check(got["y"], q4.dequant(w[1], n), a)
    assert exe.fusedMatmulNormLaunches() - before == (1 if ksplit < 2 else 0)


@pytest.mark.parametrize("over", ["sum", "norm"])
@pytest.mark.parametrize("reader", ["silu", "rope", "rope_scatter"])
def test_epilogues_over_the_norm(exe, reader, over):
    """A matmul that finishes a norm, followed by an operator that it would take over, whose output lies over the
    norm's input or output."""
    rng = np.random.default_rng(11)
    batch, n, heads, kv_heads, d = 6, 4096, 32, 4, 128
    kv = kv_heads * d
    rows = 2 * n + 64 * 2 if reader == "silu" else n + 2 * kv
    w = [_weights(rng, n, 64), _weights(rng, rows, n)]
    gamma = rng.uniform(0.5, 1.5, n).astype(np.float32)
    cos, sin = (np.stack(t) for t in zip(*(po.rotary_coefficients(int(p), d) for p in rng.integers(0, 2000, batch))))
    ids, slots = np.arange(batch, dtype=np.uint32), rng.integers(0, 8, batch).astype(np.uint32)
    half = rows // 2
    init = {"x": (batch, 64), "p": (batch, n), "r": (batch, n), "h": (batch, max(n, half)), "n": (batch, max(n, half)), "y": (batch, rows),
            "a": (batch, max(n, half)), "b": (batch, max(kv, half)), "c": (batch, max(kv, half))}
    init = {m: rng.standard_normal(s).astype(np.float32) for m, s in init.items()}
    init |= {"cos": cos.astype(np.float32), "sin": sin.astype(np.float32)}
    init |= {m: np.zeros((batch, 8, kv), np.uint16) for m in ("k16", "v16", "kp", "vp")}
    out = {}
    for fuse in (0, 1):
        dev = {m: _pool(exe, a) for m, a in init.items()}
        first = dev["h" if over == "sum" else "n"]
        assert exe.setOption("fuse_row_ops", fuse)
        before = exe.fusedMatmulNormLaunches(), exe.fusedMatmulSiluLaunches() + exe.fusedMatmulRopeLaunches()
        try:
            assert exe.beginForwardPassCB()
            assert exe.encodeMatMulQ4_0Batched("over.0", w[0], dev["x"], batch, n, 64, w[0].shape[1], 1, dev["p"]), exe.lastError()
            assert exe.encodeAddBatched(dev["r"], dev["p"], dev["h"], batch * n)
            assert exe.encodeRmsNormBatched(dev["h"], gamma, EPS, batch, n, dev["n"])
            assert exe.encodeMatMulQ4_0Batched(f"over.{reader}", w[1], dev["n"], batch, rows, n, w[1].shape[1], 1, dev["y"]), exe.lastError()
            if reader == "silu":
                assert exe.encodeGateUpSplitSiluMul(dev["y"], dev["a"], dev["b"], first, batch, half, rows), exe.lastError()
            elif reader == "rope":
                assert exe.encodeQkvSplitRopeCast(dev["y"], first, dev["b"], dev["c"], dev["k16"], dev["v16"], dev["cos"], dev["sin"],
                                                  batch, heads, kv_heads, d, rows, n, kv, kv, d), exe.lastError()
            else:
                assert exe.encodeQkvSplitRopeScatter(dev["y"], first, dev["kp"], dev["vp"], dev["cos"], dev["sin"], ids, slots, 8,
                                                     batch, heads, kv_heads, d, rows, n, kv, kv, d), exe.lastError()
            assert exe.flushForwardPassCB(), exe.lastError()
            out[fuse] = {m: _read(exe, b, init[m]) for m, b in dev.items()}
        finally:
            exe.setOption("fuse_row_ops", 1)
            for buf in dev.values():
                exe.releaseScratchBuffer(buf)
        assert exe.fusedMatmulNormLaunches() - before[0] == fuse
        assert exe.fusedMatmulSiluLaunches() + exe.fusedMatmulRopeLaunches() == before[1]
    for m, want in out[0].items():
        got = out[1][m]
        if want.dtype == np.uint16:      # fp16: one step of its rounding
            want, got = want.view(np.float16).astype(np.float32), got.view(np.float16).astype(np.float32)
        assert np.abs(got - want).max() <= (1e-3 if m in ("kp", "vp", "k16", "v16") else 1e-4) * max(np.abs(want).max(), 1e-30), m


@pytest.mark.parametrize("what", ["sum_over_gate_up", "norm_over_residual_one_row_down", "slices_sum_over_gate_up", "gate_as_residual",
                                  "slices_of_pairs_sum_over_gate_up"])
def test_row_chains_over_shared_buffers(exe, what):
    """Row operators of one chain whose buffers meet in other rows than their own: the chain's workgroups run in no order."""
    rng = np.random.default_rng(3)
    batch, n, k = 300, 1024, 512       # (more rows than run at once)
    pairs = what.startswith("slices_of_pairs")      # (the chain starts with the sum over the matmul's slices)
    if what.startswith("slices"):
        batch, k = 40, 1024 if pairs else 512
    w = _weights(rng, 2 * n, k)
    gamma = rng.uniform(0.5, 1.5, n).astype(np.float32)
    init = {"gu": (batch, 2 * n), "g": (batch, n), "u": (batch, n), "m": (batch, n), "r": (batch + 1, n), "s": (batch, n), "x": (batch, k)}
    init = {m: rng.standard_normal(s).astype(np.float32) for m, s in init.items()}
    out = {}
    for fuse in (0, 1):
        dev = {m: _pool(exe, a) for m, a in init.items()}
        assert exe.setOption("fuse_row_ops", fuse) and exe.setOption("q4_ksplit", 2) and exe.setOption("q4_int_operand", 0 if pairs else 1)
        try:
            assert exe.beginForwardPassCB()
            if what.startswith("slices"):
                assert exe.encodeMatMulQ4_0Batched(f"rows.shared.{k}", w, dev["x"], batch, 2 * n, k, w.shape[1], 1, dev["gu"]), exe.lastError()
            assert exe.encodeGateUpSplitSiluMul(dev["gu"], dev["g"], dev["u"], dev["m"], batch, n, 2 * n)
            resid, total = dev["g" if what == "gate_as_residual" else "r"], dev["gu" if "gate_up" in what else "s"]
            assert exe.encodeAddBatched(dev["m"], resid, total, batch * n)
            if "norm" in what:
                assert exe.encodeRmsNormBatched(total, gamma, EPS, batch, n, resid + 4 * n)
            assert exe.flushForwardPassCB(), exe.lastError()
            out[fuse] = {m: _read(exe, b, init[m]) for m, b in dev.items()}
        finally:
            exe.setOption("fuse_row_ops", 1)
            exe.setOption("q4_ksplit", 0)
            exe.setOption("q4_int_operand", 1)
            for buf in dev.values():
                exe.releaseScratchBuffer(buf)
    for m, want in out[0].items():
        assert np.abs(out[1][m] - want).max() <= 1e-5 * np.abs(want).max(), m
