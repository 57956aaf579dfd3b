"""Launches whose workgroups leave each other tagged words (K slices of matmuls, partials of the decode attention):
what is shared between them, the words' tags, the buffers and the order of the streams, at its limits."""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4
from oracle import paged_oracle as po
from test_matmul_norm_fusion_gpu import _pool, _read
from test_matmul_tokens_gpu import check

pytestmark = pytest.mark.gpu


def _weights(rng, rows, cols):
    return po.quantize_q4_0((rng.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float32))


def test_more_sliced_matmuls_in_a_captured_pass_than_tags(exe):
    """Those without a tag take all of K."""
    rng = np.random.default_rng(1)
    rows, cols, count = 64, 2080, 4100      # two slices each; 4096 tags
    w, x = _weights(rng, rows, cols), rng.standard_normal((1, cols)).astype(np.float32)
    d_x, d_y = _pool(exe, x), _pool(exe, np.full((count, rows), np.nan, np.float32))
    call = lambda i: exe.encodeMatMulQ4_0Batched("meet.tags", w, d_x, 1, rows, cols, w.shape[1], 1, d_y + i * rows * 4)
    handle = 0
    try:
        assert exe.beginForwardPassCB() and call(0) and exe.flushForwardPassCB(), exe.lastError()
        first = _read(exe, d_y, np.empty((count, rows), np.float32))[0]
        assert exe.beginForwardPassCB() and exe.captureBegin()
        ok = all([call(i) for i in range(count)])
        handle = exe.captureEnd()
        assert ok and handle > 0, exe.lastError()
        assert exe.flushForwardPassCB()
        for _ in range(2):
            assert exe.uploadToBuffer(d_y, np.full((count, rows), np.nan, np.float32))
            assert exe.beginForwardPassCB() and exe.replay(handle) and exe.flushForwardPassCB(), exe.lastError()
            got = _read(exe, d_y, np.empty((count, rows), np.float32))
            assert (got[:4096].view(np.uint32) == first.view(np.uint32)).all() and (got[4096:] == got[-1]).all()
            check(got[-1:], q4.dequant(w, cols), x)
    finally:
        if handle > 0:
            exe.captureRelease(handle)
        exe.releaseScratchBuffer(d_x)
        exe.releaseScratchBuffer(d_y)


def test_slices_without_room_for_their_words_in_a_captured_pass(exe):
    """Captured with more requests than have been seen: the words' buffer cannot grow, and the matmul takes all of K."""
    rng = np.random.default_rng(2)
    rows, cols = 512, 32768
    w, x = _weights(rng, rows, cols), rng.standard_normal((64, cols)).astype(np.float32)
    d_x, d_y = _pool(exe, x), exe.allocateScratchBuffer(64 * rows * 4)
    call = lambda batch: exe.encodeMatMulQ4_0Batched("meet.room", w, d_x, batch, rows, cols, w.shape[1], 1, d_y)
    handle = 0
    try:
        assert exe.setOption("q4_ksplit", 64)     # (more words than any other call needs)
        assert exe.beginForwardPassCB() and call(33) and exe.flushForwardPassCB(), exe.lastError()
        assert exe.beginForwardPassCB() and exe.captureBegin()
        ok = call(64)
        handle = exe.captureEnd()
        assert ok and handle > 0, exe.lastError()
        assert exe.flushForwardPassCB()
        for _ in range(2):
            assert exe.uploadToBuffer(d_y, np.full((64, rows), np.nan, np.float32))
            assert exe.beginForwardPassCB() and exe.replay(handle) and exe.flushForwardPassCB(), exe.lastError()
            check(_read(exe, d_y, np.empty((64, rows), np.float32)), q4.dequant(w, cols), x)
    finally:
        exe.setOption("q4_ksplit", 0)
        if handle > 0:
            exe.captureRelease(handle)
        exe.releaseScratchBuffer(d_x)
        exe.releaseScratchBuffer(d_y)
