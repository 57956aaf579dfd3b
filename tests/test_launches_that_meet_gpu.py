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


@pytest.mark.parametrize("rows,cols,batch", [(64, 4096, 5), (4160, 2080, 1000)])
def test_the_decode_spin_limit_is_not_the_matmuls(exe, rows, cols, batch):
    """A matmul waits for its slices as long as ever where the decode attention's wait is cut short."""
    rng = np.random.default_rng(3)
    w, x = _weights(rng, rows, cols), rng.standard_normal((batch, cols)).astype(np.float32)
    d_x, d_y = _pool(exe, x), exe.allocateScratchBuffer(batch * rows * 4)
    try:
        assert exe.setOption("decode_spin_limit", 1)
        for _ in range(20):
            assert exe.encodeMatMulQ4_0Batched("meet.spin", w, d_x, batch, rows, cols, w.shape[1], 1, d_y, True), exe.lastError()
        check(_read(exe, d_y, np.empty((batch, rows), np.float32)), q4.dequant(w, cols), x)
    finally:
        exe.setOption("decode_spin_limit", 200000)
        exe.releaseScratchBuffer(d_x)
        exe.releaseScratchBuffer(d_y)


MEMORY = """
import ctypes as C, numpy as np, sys
sys.path[:0] = ["tests", "."]
from mlcompiler_amd import HipExecutor
import test_q4_matmul_gpu as q4
exe, hip = HipExecutor.Instance(), C.CDLL("libamdhip64.so")
exe.requireAvailable()
used = []
# 80 tiles, too short to be split; 128 and 32 tiles left over by whole rounds, too short and long enough
for rows, cols, tokens in ((64, 256, 5120), (4096, 960, 1030), (4096, 1024, 1030)):
    q, x, stride = q4.make(rows, cols, tokens, rows)
    q4.run(exe, f"memory_{rows}_{cols}", q, x, tokens, rows, cols, stride)
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    used.append(total.value - free.value)
print("used", *used)
"""


def test_only_split_tiles_take_memory_to_meet_in():
    """(A process of its own: the library's buffers are for good.)"""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", MEMORY], cwd=root, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    first, whole, split = (int(v) >> 20 for v in out.stdout.split("used")[1].split())
    print(f"in use: {first}, {whole}, {split} MiB")
    assert whole - first < 32 <= split - whole


def _decode(exe):
    """A decode attention whose pairs are split over workgroups."""
    from paged_cases import DeviceCase, baseline_config
    case = baseline_config(2, batch=6)
    dev = DeviceCase(exe, case)
    out = np.empty((case.batch, case.num_heads, case.head_dim), np.float32)
    call = lambda: exe.encodePagedFlashAttention(dev.q_buf, dev.k_buf, dev.v_buf, dev.o_buf, case.page_tables_flat, case.page_table_offsets,
                                                 case.seq_lens, case.q_positions, case.batch, case.num_heads, case.kv_heads,
                                                 case.head_dim, case.page_size, case.apply_causal)
    return call, lambda: _read(exe, dev.o_buf, out), dev.free


def _matmul(rows, cols, batch):
    def make(exe):
        rng = np.random.default_rng(rows)
        w, x = _weights(rng, rows, cols), rng.standard_normal((batch, cols)).astype(np.float32)
        d_x, d_y = _pool(exe, x), exe.allocateScratchBuffer(batch * rows * 4)
        call = lambda: exe.encodeMatMulQ4_0Batched(f"meet.{rows}.{cols}", w, d_x, batch, rows, cols, w.shape[1], 1, d_y)
        return call, lambda: _read(exe, d_y, np.empty((batch, rows), np.float32)), lambda: [exe.releaseScratchBuffer(b) for b in (d_x, d_y)]
    return make


KINDS = {"decode": _decode, "slices": _matmul(64, 4096, 5), "tail": _matmul(4160, 1024, 1000)}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("captured", [False, True])
def test_tags_that_come_again(exe, kind, captured):
    """Every launch (replay) takes more than half of the tags, so that they start over at once, and the second one does not write
    its words: those of the first, which had the same tag, are gone, and the wait for the second's is given up."""
    call, read, free = KINDS[kind](exe)
    handles = []

    def run(flags):
        assert exe.setOption("decode_test_flags", flags) and exe.setOption("decode_spin_limit", 3 if flags & 1 else 200000)
        if captured:
            assert exe.beginForwardPassCB() and exe.captureBegin()
            assert call(), exe.lastError()
            handles.append(exe.captureEnd())
            assert handles[-1] > 0 and exe.flushForwardPassCB(), exe.lastError()
            assert exe.beginForwardPassCB() and exe.replay(handles[-1]), exe.lastError()
        else:
            assert exe.beginForwardPassCB() and call(), exe.lastError()
        return exe.flushForwardPassCB()

    try:
        assert run(0) if not captured else (exe.beginForwardPassCB() and call() and exe.flushForwardPassCB()), exe.lastError()
        want = read()
        for _ in range(3):
            assert run(2), exe.lastError()
            assert np.array_equal(read(), want)
        assert not run(3) and "gave up" in exe.lastError()
        for _ in range(3):
            assert run(0), exe.lastError()
            assert np.array_equal(read(), want)
    finally:
        exe.setOption("decode_test_flags", 0)
        exe.setOption("decode_spin_limit", 200000)
        for h in handles:
            exe.captureRelease(h)
        free()


def _hip():
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")
    for name in ("hipStreamCreate", "hipStreamSynchronize", "hipStreamDestroy", "hipStreamQuery", "hipMemcpyAsync"):
        getattr(hip, name).argtypes = {"hipStreamCreate": [C.POINTER(C.c_void_p)],
                                       "hipMemcpyAsync": [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]}.get(name, [C.c_void_p])
    return hip


@pytest.mark.parametrize("kind", ["slices", "tail", "replayed"])
def test_waiting_launches_on_two_streams_follow_each_other(exe, kind):
    """A matmul whose slices meet and a decode attention on a caller's stream: side by side, each could hold the CUs
    that workgroups need for which the other one's wait."""
    import ctypes as C
    from mlcompiler_amd._lib import load
    from paged_cases import DeviceCase, baseline_config
    lib, hip, stream = load(), _hip(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    library = C.c_void_p(lib.mlc_hip_stream())
    call, read, free = KINDS["tail" if kind == "tail" else "slices"](exe)
    case = baseline_config(2, batch=6)
    dev = DeviceCase(exe, case)
    arrays = [np.ascontiguousarray(a, np.uint32) for a in (case.page_tables_flat, case.page_table_offsets, case.seq_lens, case.q_positions)]
    d_flat = _pool(exe, arrays[0])
    u32p = lambda a: a.ctypes.data_as(C.POINTER(C.c_uint32))
    big = 1 << 28
    d_a, d_b = exe.allocateScratchBuffer(big), exe.allocateScratchBuffer(big)
    handle = 0

    def decode():
        return lib.mlc_hip_paged_attn_decode_noalloc(dev.q_buf, dev.k_buf, dev.v_buf, dev.o_buf, d_flat, arrays[0].size, u32p(arrays[1]),
                                                     u32p(arrays[2]), u32p(arrays[3]), case.batch, case.num_heads, case.kv_heads,
                                                     case.head_dim, case.page_size, int(case.apply_causal), stream)

    def busy(s):     # some milliseconds of copies
        for _ in range(40):
            assert hip.hipMemcpyAsync(d_a, d_b, big, 3, s) == 0
        assert hip.hipStreamQuery(s) == 600      # (not ready)

    try:
        want_o = dev.run()
        assert exe.setOption("fuse_row_ops", 0)      # (nothing held back: that orders the streams by itself)
        assert exe.beginForwardPassCB() and call() and exe.flushForwardPassCB(), exe.lastError()
        want = read()
        if kind == "replayed":
            assert exe.beginForwardPassCB() and exe.captureBegin() and call()
            handle = exe.captureEnd()
            assert handle > 0 and exe.flushForwardPassCB(), exe.lastError()
        launch = (lambda: exe.replay(handle)) if handle else call
        # a matmul behind the other stream's decode
        busy(stream)
        assert decode(), exe.lastError()
        assert exe.beginForwardPassCB() and launch() and exe.flushForwardPassCB(), exe.lastError()
        assert hip.hipStreamQuery(stream) == 0
        assert np.array_equal(read(), want)
        # and the decode behind the matmul
        busy(library)
        assert exe.beginForwardPassCB() and launch(), exe.lastError()
        assert decode(), exe.lastError()
        assert hip.hipStreamSynchronize(stream) == 0 and hip.hipStreamQuery(library) == 0
        assert exe.flushForwardPassCB(), exe.lastError()
        assert np.array_equal(read(), want)
        assert np.array_equal(_read(exe, dev.o_buf, want_o), want_o)
    finally:
        exe.setOption("fuse_row_ops", 1)
        if handle > 0:
            exe.captureRelease(handle)
        hip.hipStreamSynchronize(stream)
        hip.hipStreamDestroy(stream)
        for b in (d_flat, d_a, d_b):
            exe.releaseScratchBuffer(b)
        dev.free()
        free()


def test_a_decode_recorded_into_a_callers_graph_orders_nothing(exe):
    """It does not run when it is recorded: the library's launches behind it neither wait for it nor fail."""
    import ctypes as C
    from mlcompiler_amd._lib import load
    from paged_cases import DeviceCase, baseline_config
    lib, hip, stream, graph = load(), _hip(), C.c_void_p(), C.c_void_p()
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphDestroy.argtypes = [C.c_void_p]
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    call, read, free = KINDS["slices"](exe)
    case = baseline_config(2, batch=6)
    dev = DeviceCase(exe, case)
    arrays = [np.ascontiguousarray(a, np.uint32) for a in (case.page_tables_flat, case.page_table_offsets, case.seq_lens, case.q_positions)]
    d_flat = _pool(exe, arrays[0])
    u32p = lambda a: a.ctypes.data_as(C.POINTER(C.c_uint32))
    try:
        want_o = dev.run()
        assert exe.beginForwardPassCB() and call() and exe.flushForwardPassCB(), exe.lastError()
        want = read()
        assert hip.hipStreamBeginCapture(stream, 1) == 0       # (this thread's calls)
        ok = lib.mlc_hip_paged_attn_decode_noalloc(dev.q_buf, dev.k_buf, dev.v_buf, dev.o_buf, d_flat, arrays[0].size, u32p(arrays[1]),
                                                   u32p(arrays[2]), u32p(arrays[3]), case.batch, case.num_heads, case.kv_heads,
                                                   case.head_dim, case.page_size, int(case.apply_causal), stream)
        ended = hip.hipStreamEndCapture(stream, C.byref(graph))
        assert ok and ended == 0 and graph, exe.lastError()
        assert hip.hipGraphDestroy(graph) == 0
        assert exe.beginForwardPassCB() and call() and exe.flushForwardPassCB(), exe.lastError()
        assert np.array_equal(read(), want) and np.array_equal(dev.run(), want_o)
    finally:
        hip.hipStreamDestroy(stream)
        exe.releaseScratchBuffer(d_flat)
        dev.free()
        free()


@pytest.mark.parametrize("own", [True, False])      # a stream of the caller's, or the library's
@pytest.mark.parametrize("flags", [0, 2])
def test_a_decode_replayed_from_a_callers_graph(exe, flags, own):
    """Every replay sums the partials of its own, and none of the one before (at once also where the tags start over)."""
    import ctypes as C
    from mlcompiler_amd._lib import load
    from paged_cases import DeviceCase, baseline_config
    lib, hip, stream, graph, run = load(), _hip(), C.c_void_p(), C.c_void_p(), C.c_void_p()
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    hip.hipGraphExecDestroy.argtypes = hip.hipGraphDestroy.argtypes = [C.c_void_p]
    case = baseline_config(2, batch=6)
    dev = DeviceCase(exe, case)
    arrays = [np.ascontiguousarray(a, np.uint32) for a in (case.page_tables_flat, case.page_table_offsets, case.seq_lens, case.q_positions)]
    d_flat, d_o = _pool(exe, arrays[0]), exe.allocateScratchBuffer(case.q.nbytes)
    u32p = lambda a: a.ctypes.data_as(C.POINTER(C.c_uint32))
    rng = np.random.default_rng(4)
    qs = [rng.standard_normal(case.q.shape).astype(np.float32) for _ in range(20)]
    want = []
    if own:
        assert hip.hipStreamCreate(C.byref(stream)) == 0
    else:
        stream.value = lib.mlc_hip_stream()
    try:
        for q in qs:
            assert exe.uploadToBuffer(dev.q_buf, q)
            want.append(dev.run().copy())
        assert exe.setOption("decode_test_flags", flags)
        assert hip.hipStreamBeginCapture(stream, 1) == 0       # (this thread's calls)
        ok = lib.mlc_hip_paged_attn_decode_noalloc(dev.q_buf, dev.k_buf, dev.v_buf, d_o, d_flat, arrays[0].size, u32p(arrays[1]),
                                                   u32p(arrays[2]), u32p(arrays[3]), case.batch, case.num_heads, case.kv_heads,
                                                   case.head_dim, case.page_size, int(case.apply_causal), stream)
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and ok, exe.lastError()
        assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
        assert exe.setOption("decode_test_flags", 0)
        for q, o in zip(qs, want):
            assert exe.uploadToBuffer(dev.q_buf, q)
            assert hip.hipGraphLaunch(run, stream) == 0 and hip.hipStreamSynchronize(stream) == 0
            assert np.array_equal(_read(exe, d_o, np.empty_like(o)), o)
    finally:
        exe.setOption("decode_test_flags", 0)
        if run:
            hip.hipGraphExecDestroy(run)
        if graph:
            hip.hipGraphDestroy(graph)
        if own:
            hip.hipStreamDestroy(stream)
        for b in (d_flat, d_o):
            exe.releaseScratchBuffer(b)
        dev.free()
