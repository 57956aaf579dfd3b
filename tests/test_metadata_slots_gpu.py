"""Calls whose tables go through the library's pinned slots: encoding more of them than there are slots neither
empties the queue nor writes a slot that a launch still reads."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

B, M, H, KV, D, P, CTX, CALLS = 8, 1024, 32, 8, 128, 64, 8192, 9   # one call more than slots; about 2 ms of work each


def test_the_ninth_call_does_not_wait_for_the_eighth(exe):
    rng = np.random.default_rng(1)
    pages = (CTX + M) // P
    assert 3 * B + B * pages > 960                       # more words than travel inside the arguments
    pool = B * pages
    off = (np.arange(B + 1) * pages).astype(np.uint32)
    seq, start = np.full(B, CTX + M, np.uint32), np.full(B, CTX, np.uint32)
    row = KV * D * 2
    sizes = dict(q=B * M * H * D * 2, k=pool * P * row, v=pool * P * row)
    buf = {n: exe.allocateScratchBuffer(s) for n, s in sizes.items()}
    outs = [exe.allocateScratchBuffer(B * M * H * D * 4) for _ in range(CALLS)]
    tables = [rng.permutation(pool).astype(np.uint32) for _ in range(CALLS)]

    def call(i, encode):
        assert exe.runPagedPrefillAttention(buf["q"], buf["k"], buf["v"], outs[i], tables[i], off, seq, start, B, M, H, KV, D, P,
                                            sync=not encode), exe.lastError()

    def result(i):
        o = np.empty((B, M, H * D), np.float32)
        assert exe.downloadFromBuffer(outs[i], o)
        return o[:, ::64].copy()

    try:
        for n, s in sizes.items():
            assert exe.uploadToBuffer(buf[n], rng.standard_normal(s // 2, dtype=np.float32).astype(np.float16))
        want, took = [], []
        for i in range(CALLS):
            t0 = time.perf_counter()
            call(i, False)
            took.append(time.perf_counter() - t0)
            want.append(result(i))
            assert exe.zeroBuffer(outs[i], B * M * H * D * 4)
        assert exe.beginForwardPassCB()
        for i in range(CALLS):
            call(i, True)
        t0 = time.perf_counter()
        assert exe.flushForwardPassCB(), exe.lastError()
        left = time.perf_counter() - t0
        for i in range(CALLS):
            assert np.array_equal(result(i), want[i]), f"call {i}"
        print(f"[slots] one call {1e3 * np.median(took):.2f} ms, left behind the last encode {1e3 * left:.2f} ms")
        assert left > 3.5 * np.median(took)              # (all but the oldest two or so are still to come)
    finally:
        for b in (*buf.values(), *outs):
            exe.releaseScratchBuffer(b)
