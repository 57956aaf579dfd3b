"""Q4_0 and Q6_K matmuls over more than 64 tokens (one launch for all of them) against a float64
product of the dequantised weights: the edges of the kernel's tiles (64 tokens, 128 rows, stages of 64
columns, turns of 4 stages), K split over workgroups or not, and inputs larger than one piece.

Tolerance per output element, relative to A = sum_c |w_c * x_c|: as for the kernels that take 64 requests
at a time, 4e-6 (activations as fp16 pairs: 2^-22 per product; fp32 sums)."""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4
import test_q6k_matmul_gpu as q6
from oracle import paged_oracle as po

pytestmark = pytest.mark.gpu


def check(got, w, x):
    w, x = w.astype(np.float64), x.astype(np.float64)
    err = np.max(np.abs(got - x @ w.T) / (np.abs(x) @ np.abs(w).T + 1e-30))
    print(f"  max |got-exact|/A = {err:.2e}", flush=True)
    assert err < 4e-6


@pytest.mark.parametrize("rows,cols,tokens", [
    (64, 64, 65),         # one stage, half a row block, the first token of the second token block
    (128, 96, 127),       # an odd number of blocks
    (192, 160, 128), (320, 288, 129),
    (64, 2048, 64 * 9 + 1),        # a second group of token blocks, K split
    (2048, 4096, 70),     # K split as far as it goes
    (8192, 320, 300),     # more workgroups than fit at once, K whole
    (64, 14336, 1153),    # one token more than a piece holds
])
def test_q4_tokens(exe, rows, cols, tokens):
    print(f"[q4 tokens] rows={rows} cols={cols} tokens={tokens}", flush=True)
    q, x, stride = q4.make(rows, cols, tokens, rows + cols + tokens)
    x[tokens // 2] = 0.0
    got = q4.run(exe, f"tok4_{rows}_{cols}", q, x, tokens, rows, cols, stride)
    assert np.all(got[tokens // 2] == 0.0)
    check(got, q4.dequant(q, cols), x)
    assert np.array_equal(got, q4.run(exe, f"tok4_{rows}_{cols}", q, x, tokens, rows, cols, stride, sync=False))


@pytest.mark.parametrize("rows,cols,tokens", [(32, 256, 65), (96, 512, 128), (160, 2048, 577), (4128, 768, 200)])
def test_q6k_tokens(exe, rows, cols, tokens):
    print(f"[q6k tokens] rows={rows} cols={cols} tokens={tokens}", flush=True)
    q, x, stride = q6.make(rows, cols, tokens, rows + cols + tokens)
    got = q6.run(exe, f"tok6_{rows}_{cols}", q, x, tokens, rows, cols, stride)
    check(got, po.dequantize_q6_k(np.ascontiguousarray(q[:, :po.q6_k_row_bytes(cols)]), cols), x)


def test_tokens_pass_replayed(exe):
    # recorded into a graph (a split of K among its launches) and replayed between eager calls
    rows, cols, tokens = 256, 2048, 100
    q, x, stride = q4.make(rows, cols, tokens, 7)
    eager = q4.run(exe, "tok_replay", q, x, tokens, rows, cols, stride)
    d_in, d_out = exe.allocateScratchBuffer(x.nbytes), exe.allocateScratchBuffer(tokens * rows * 4)
    assert exe.uploadToBuffer(d_in, x)
    assert exe.beginForwardPassCB() and exe.captureBegin()
    assert exe.encodeMatMulQ4_0Batched("tok_replay", q, d_in, tokens, rows, cols, stride, 1, d_out), exe.lastError()
    handle = exe.captureEnd()
    try:
        assert handle > 0, exe.lastError()
        assert exe.flushForwardPassCB()
        for _ in range(3):
            assert exe.uploadToBuffer(d_out, np.full(tokens * rows, np.nan, np.float32))
            assert exe.beginForwardPassCB() and exe.replay(handle) and exe.flushForwardPassCB()
            got = np.empty((tokens, rows), np.float32)
            assert exe.downloadFromBuffer(d_out, got)
            assert np.array_equal(got, eager)
            q4.run(exe, "tok_replay", q, -x[:70], 70, rows, cols, stride)
    finally:
        exe.captureRelease(handle)
        exe.releaseScratchBuffer(d_in)
        exe.releaseScratchBuffer(d_out)
