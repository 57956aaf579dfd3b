"""A captured pass finds the page rows of its KV write on the device whichever way the uncaptured pass before
it passed them: inside the kernel arguments or, for more requests than those hold, already on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H, KV, D, P = 4, 2, 64, 16
ROW = KV * D
QKV = (H + 2 * KV) * D


@pytest.mark.parametrize("B", [1, 64, 65, 256, 257])   # around the rows that a rotation's and a scatter's arguments hold
def test_capture_right_after_an_uncaptured_pass(exe, B):
    rng = np.random.default_rng(B)
    pool = np.zeros(B * P * ROW, np.uint16)
    names = dict(qkv=B * QKV * 4, q=B * H * D * 4, k=B * ROW * 4, v=B * ROW * 4, k16=B * ROW * 2, v16=B * ROW * 2,
                 cos=B * D * 2, sin=B * D * 2, kp=pool.nbytes, vp=pool.nbytes)
    buf = {n: exe.allocateScratchBuffer(s) for n, s in names.items()}
    handle = 0
    other, ids, later = (rng.permutation(B).astype(np.uint32) for _ in range(3))
    slots = rng.integers(0, P, B).astype(np.uint32)
    zero = np.zeros(0, np.uint32)

    def scatters(page_ids):
        for pages, rows in (("kp", "k16"), ("vp", "v16")):
            assert exe.encodeScatterKVPagedBatched(buf[pages], page_ids, slots, P, KV, D, B, buf[rows]), exe.lastError()

    def step(page_ids):
        assert exe.encodeQkvSplitRopeCast(buf["qkv"], buf["q"], buf["k"], buf["v"], buf["k16"], buf["v16"], buf["cos"], buf["sin"],
                                          B, H, KV, D, QKV, H * D, ROW, ROW, D), exe.lastError()
        scatters(page_ids)

    def pools():
        out = [np.empty_like(pool) for _ in range(2)]
        assert exe.downloadFromBuffer(buf["kp"], out[0]) and exe.downloadFromBuffer(buf["vp"], out[1])
        return out

    def cleared():
        assert exe.zeroBuffer(buf["kp"], pool.nbytes) and exe.zeroBuffer(buf["vp"], pool.nbytes)

    try:
        for n in ("qkv", "cos", "sin"):
            assert exe.uploadToBuffer(buf[n], rng.standard_normal(names[n] // 4, dtype=np.float32))
        cleared()
        assert exe.beginForwardPassCB()
        scatters(other)                                  # rows of another pass of the same size
        assert exe.flushForwardPassCB(), exe.lastError()
        cleared()
        assert exe.beginForwardPassCB()
        step(ids)
        assert exe.flushForwardPassCB(), exe.lastError()
        want = pools()
        assert exe.beginForwardPassCB() and exe.captureBegin(), exe.lastError()
        step(ids)
        handle = exe.captureEnd()
        assert handle > 0, exe.lastError()
        assert exe.flushForwardPassCB(), exe.lastError()
        for page_ids in (ids, later, ids):
            cleared()
            assert exe.replayUpdate(handle, zero, np.zeros(1, np.uint32), np.zeros(B, np.uint32), zero, page_ids, slots), exe.lastError()
            assert exe.beginForwardPassCB() and exe.replay(handle) and exe.flushForwardPassCB(), exe.lastError()
            got = pools()
            if page_ids is ids:
                assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
            else:
                rows = [p.reshape(B, P, ROW) for p in (*got, *want)]
                for r in range(B):
                    assert np.array_equal(rows[0][later[r], slots[r]], rows[2][ids[r], slots[r]])
                    assert np.array_equal(rows[1][later[r], slots[r]], rows[3][ids[r], slots[r]])
    finally:
        if handle:
            exe.captureRelease(handle)
        for b in buf.values():
            exe.releaseScratchBuffer(b)
