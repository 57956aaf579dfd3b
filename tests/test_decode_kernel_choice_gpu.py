"""Which kernel a decode call gets depends on its shape and the options alone, never on the lengths of the moment:
a replayed pass and the same step encoded call by call give the same bits however far the contexts have grown."""
import numpy as np
import pytest

from paged_cases import DeviceCase, assert_parity, make_case, oracle_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("ratio", [1, 2, 3, 4])
def test_replay_at_longer_contexts_equals_the_eager_call(exe, D, ratio):
    short, long = [3, 70, 40], [2900, 1500, 2222]
    c = make_case(f"grow_{ratio}_{D}", 3, 8 * ratio, 8, D, 64, long, seed=ratio)
    dev = DeviceCase(exe, c)
    args = (dev.q_buf, dev.k_buf, dev.v_buf, dev.o_buf, c.page_tables_flat, c.page_table_offsets)
    shape = (c.batch, c.num_heads, c.kv_heads, D, 64, True)
    handle = 0

    def encode(lens):
        seq = np.array(lens, np.uint32)
        assert exe.encodePagedFlashAttention(*args, seq, seq - 1, *shape), exe.lastError()

    def output():
        o = np.empty_like(c.q)
        assert exe.downloadFromBuffer(dev.o_buf, o)
        return o

    try:
        assert exe.beginForwardPassCB()
        encode(short)
        assert exe.flushForwardPassCB(), exe.lastError()
        at_short = exe.lastDecodeKernel()
        assert exe.beginForwardPassCB() and exe.captureBegin(), exe.lastError()
        encode(short)
        handle = exe.captureEnd()
        assert handle > 0, exe.lastError()
        assert exe.flushForwardPassCB()
        assert exe.beginForwardPassCB()
        encode(long)
        assert exe.flushForwardPassCB(), exe.lastError()
        want = output()
        assert exe.lastDecodeKernel() == at_short
        seq = np.array(long, np.uint32)
        for _ in range(3):
            assert exe.replayUpdate(handle, c.page_tables_flat, c.page_table_offsets, seq, seq - 1), exe.lastError()
            assert exe.beginForwardPassCB() and exe.replay(handle) and exe.flushForwardPassCB(), exe.lastError()
            assert np.array_equal(output(), want)
    finally:
        if handle:
            exe.captureRelease(handle)
        dev.free()
