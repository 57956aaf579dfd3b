"""Q4_0 matmuls whose K is split over workgroups: the slices leave their sums as tagged words and the last one's
workgroups add them up inside the launch."""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4
from oracle import paged_oracle as po
from test_matmul_norm_fusion_gpu import EPS, _pool, _read
from test_matmul_tokens_gpu import check

pytestmark = pytest.mark.gpu


def _weights(rng, rows, cols):
    return po.quantize_q4_0((rng.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float32))


# three slices of 44 quads, two groups of requests, an incomplete last quad, one group of many slices, one tile per workgroup
SHAPES = [(2048, 5632, 1), (2048, 5632, 8), (2048, 5632, 21), (128, 2080, 16), (64, 14336, 5), (64, 4096, 64), (4096, 14336, 49)]


@pytest.mark.parametrize("rows,cols,batch", SHAPES)
@pytest.mark.parametrize("behind", ["nothing", "add", "add_in_place", "norm"])
def test_slices_meet(exe, rows, cols, batch, behind):
    """The same bits on every run, with the operators behind the matmul in its epilogue or not."""
    rng = np.random.default_rng(rows + cols + batch)
    w, w2 = _weights(rng, rows, cols), _weights(rng, 4096, rows)
    x, r = (rng.standard_normal((batch, n)).astype(np.float32) for n in (cols, rows))
    gamma = (1.0 + 0.3 * rng.standard_normal(rows)).astype(np.float32)
    like = {"p": np.empty((batch, rows), np.float32), "h": np.empty((batch, rows), np.float32),
            "n": np.empty((batch, rows), np.float32), "y": np.empty((batch, 4096), np.float32)}
    out = []
    for fuse in (1, 1, 0):
        dev = {m: _pool(exe, np.full_like(a, np.nan)) for m, a in like.items()}
        d_x, d_r = _pool(exe, x), _pool(exe, r)
        if behind == "add_in_place":
            exe.releaseScratchBuffer(dev["h"])
            dev["h"] = d_r
        assert exe.setOption("fuse_row_ops", fuse)
        try:
            assert exe.beginForwardPassCB()
            assert exe.encodeMatMulQ4_0Batched(f"slices.{rows}.{cols}.{batch}", w, d_x, batch, rows, cols, w.shape[1], 1, dev["p"]), exe.lastError()
            if behind != "nothing":
                assert exe.encodeAddBatched(dev["p"], d_r, dev["h"], batch * rows), exe.lastError()
            if behind == "norm":
                assert exe.encodeRmsNormBatched(dev["h"], gamma, EPS, batch, rows, dev["n"]), exe.lastError()
                assert exe.encodeMatMulQ4_0Batched(f"slices.{rows}.{cols}.{batch}.2", w2, dev["n"], batch, 4096, rows, w2.shape[1], 1,
                                                   dev["y"]), exe.lastError()
            assert exe.flushForwardPassCB(), exe.lastError()
            out.append({m: _read(exe, b, like[m]) for m, b in dev.items()})
        finally:
            exe.setOption("fuse_row_ops", 1)
            for buf in {*dev.values(), d_x, d_r}:
                exe.releaseScratchBuffer(buf)
    for m in like:
        assert np.array_equal(out[0][m].view(np.uint32), out[1][m].view(np.uint32)), m
    got = out[0]
    check(got["p"], q4.dequant(w, cols), x)
    assert np.array_equal(got["p"].view(np.uint32), out[2]["p"].view(np.uint32))
    if behind != "nothing":
        assert np.array_equal(got["h"], r + got["p"])
    if behind == "norm":
        want = po.rms_norm_batched(got["h"], gamma, EPS, batch, rows)
        assert (np.abs(got["n"] - want) <= 2e-6 * np.abs(want).max(axis=1, keepdims=True)).all()
        check(got["y"], q4.dequant(w2, rows), got["n"])


def test_slices_in_a_captured_pass(exe):
    """Every replay, with eager matmuls over the same words between them, gives what its own input asks for."""
    rng = np.random.default_rng(5)
    batch, rows, cols = 6, 256, 8192
    w = [_weights(rng, rows, cols) for _ in range(3)]
    dense = [q4.dequant(a, cols) for a in w]
    d_x, d_e = (exe.allocateScratchBuffer(batch * n * 4) for n in (cols, rows))
    d_y = [exe.allocateScratchBuffer(batch * rows * 4) for _ in w]

    def encode():
        for i, y in enumerate(d_y):
            assert exe.encodeMatMulQ4_0Batched(f"replayed.{i}", w[i], d_x, batch, rows, cols, w[i].shape[1], 1, y), exe.lastError()

    handle = 0
    try:
        assert exe.uploadToBuffer(d_x, np.zeros((batch, cols), np.float32))
        assert exe.beginForwardPassCB()
        encode()
        assert exe.flushForwardPassCB()
        assert exe.beginForwardPassCB() and exe.captureBegin()
        encode()
        handle = exe.captureEnd()
        assert handle > 0 and exe.flushForwardPassCB(), exe.lastError()
        for turn in range(6):
            x = rng.standard_normal((batch, cols)).astype(np.float32)
            assert exe.uploadToBuffer(d_x, x)
            assert exe.beginForwardPassCB() and exe.replay(handle) and exe.flushForwardPassCB(), exe.lastError()
            got = [_read(exe, y, np.empty((batch, rows), np.float32)) for y in d_y]
            assert exe.encodeMatMulQ4_0Batched(f"replayed.{turn % 3}", w[turn % 3], d_x, batch, rows, cols, w[0].shape[1], 1, d_e, True)
            eager = _read(exe, d_e, got[0])
            assert np.array_equal(eager.view(np.uint32), got[turn % 3].view(np.uint32))
            for a, b in zip(got, dense):
                check(a, b, x)
    finally:
        if handle > 0:
            exe.captureRelease(handle)
        for buf in [d_x, d_e, *d_y]:
            exe.releaseScratchBuffer(buf)


def test_a_slice_that_never_comes(exe):
    """The bounded wait ends, the pass fails, and the next one works."""
    rng = np.random.default_rng(6)
    batch, rows, cols = 3, 64, 4096
    w, x = _weights(rng, rows, cols), rng.standard_normal((batch, cols)).astype(np.float32)
    d_x, d_y = _pool(exe, x), exe.allocateScratchBuffer(batch * rows * 4)
    call = lambda: exe.encodeMatMulQ4_0Batched("never", w, d_x, batch, rows, cols, w.shape[1], 1, d_y, True)
    try:
        assert call()
        assert exe.setOption("decode_test_flags", 1) and exe.setOption("decode_spin_limit", 3)
        assert not call() and "gave up" in exe.lastError()
        assert exe.setOption("decode_test_flags", 0) and exe.setOption("decode_spin_limit", 200000)
        assert call()
        check(_read(exe, d_y, np.empty((batch, rows), np.float32)), q4.dequant(w, cols), x)
    finally:
        exe.setOption("decode_test_flags", 0)
        exe.setOption("decode_spin_limit", 200000)
        exe.releaseScratchBuffer(d_x)
        exe.releaseScratchBuffer(d_y)
