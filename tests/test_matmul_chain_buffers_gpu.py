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
    # 512 workgroups of 16 waves, one to a CU, in the middle: its second half starts when the first has written the
    # next input, which is wider than its own
    (64, (64, 2048, 4096, 8192), 2),
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
