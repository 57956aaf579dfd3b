"""Matmuls over many tokens whose workgroups leave a part of their last round: those tiles' K is split over workgroups that meet
inside the launch.  (Sizes for 256 CUs, 512 workgroups at a time; on another part they are ordinary sizes.)"""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4
import test_q6k_matmul_gpu as q6
from oracle import paged_oracle as po
from test_matmul_tokens_gpu import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,rows,cols,tokens", [
    ("q4", 4160, 2080, 1000),    # 16 tiles left, three slices, the last one shorter; half of the last row block missing
    ("q4", 4096, 1024, 1030),    # 32 left, two slices, tokens missing in the last block
    ("q4", 8192, 2752, 640),     # 128 left, four slices: every slot taken
    ("q4", 8192, 2688, 640),     # ... K too short for so many
    ("q4", 6144, 1024, 1024),    # 256 left: none split
    ("q4", 4096, 960, 1030),     # too short to be split
    ("q4", 2048, 2048, 500),     # all 128 tiles in four slices
    ("q4", 6144, 2080, 300),     # 240 tiles in two, the second one shorter
    ("q6", 4128, 768, 200),      # 132 tiles in three
    ("q6", 4128, 2048, 1000), ("q6", 6144, 1024, 700),
    ("q4", 4160, 4160, 1000),    # 65 stages, 20 in a slice: first-level sums of 8, by the whole K, the slice's last one shorter
    ("q4", 4096, 7232, 1030),    # 113 stages
    ("q6", 4128, 4352, 1000),    # 68
])
def test_tail(exe, fmt, rows, cols, tokens):
    print(f"[tokens tail] {fmt} rows={rows} cols={cols} tokens={tokens}", flush=True)
    m = q4 if fmt == "q4" else q6
    q, x, stride = m.make(rows, cols, tokens, rows + cols + tokens)
    w = q4.dequant(q, cols) if fmt == "q4" else po.dequantize_q6_k(np.ascontiguousarray(q[:, :po.q6_k_row_bytes(cols)]), cols)
    got = m.run(exe, f"tail_{fmt}_{rows}_{cols}", q, x, tokens, rows, cols, stride)
    check(got, w, x)
    assert np.array_equal(got, m.run(exe, f"tail_{fmt}_{rows}_{cols}", q, x, tokens, rows, cols, stride))


def test_tail_replayed(exe):
    rows, cols, tokens = 4160, 1024, 1000
    q, x, stride = q4.make(rows, cols, tokens, 8)
    eager = q4.run(exe, "tail_replay", q, x, tokens, rows, cols, stride)
    d_in, d_out = exe.allocateScratchBuffer(x.nbytes), exe.allocateScratchBuffer(tokens * rows * 4)
    assert exe.uploadToBuffer(d_in, x)
    assert exe.beginForwardPassCB() and exe.captureBegin()
    assert exe.encodeMatMulQ4_0Batched("tail_replay", q, d_in, tokens, rows, cols, stride, 1, d_out), exe.lastError()
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
            q4.run(exe, "tail_replay", q, -x, tokens, rows, cols, stride)
    finally:
        exe.captureRelease(handle)
        exe.releaseScratchBuffer(d_in)
        exe.releaseScratchBuffer(d_out)


@pytest.mark.parametrize("rows,cols,tokens", [(4160, 1024, 1000), (2048, 2048, 500)])    # a tail; all tiles
def test_a_slice_that_never_comes(exe, rows, cols, tokens):
    """The bounded wait ends, the pass fails, and the next one works."""
    q, x, stride = q4.make(rows, cols, tokens, 9)
    d_in, d_out = exe.allocateScratchBuffer(x.nbytes), exe.allocateScratchBuffer(tokens * rows * 4)
    call = lambda: exe.encodeMatMulQ4_0Batched(f"tail_never_{rows}", q, d_in, tokens, rows, cols, stride, 1, d_out, True)
    try:
        assert exe.uploadToBuffer(d_in, x) and call()
        assert exe.setOption("decode_test_flags", 1) and exe.setOption("decode_spin_limit", 3)
        assert not call() and "gave up" in exe.lastError()
        assert exe.setOption("decode_test_flags", 0) and exe.setOption("decode_spin_limit", 200000)
        assert call()
        got = np.empty((tokens, rows), np.float32)
        assert exe.downloadFromBuffer(d_out, got)
        check(got, q4.dequant(q, cols), x)
    finally:
        exe.setOption("decode_test_flags", 0)
        exe.setOption("decode_spin_limit", 200000)
        exe.releaseScratchBuffer(d_in)
        exe.releaseScratchBuffer(d_out)
