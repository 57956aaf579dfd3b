"""Q4_0 matmuls that are a call of their own over up to eight requests split their rows of floats themselves: row tiles per
workgroup, quads that end early, K slices, the requests where another launch splits them instead, and rows whose blocks are far apart."""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("rows,cols", [
    (64, 64), (192, 96),            # half a quad; three blocks
    (2048, 2080),                   # slices, the last of them with a quad of one block
    (256, 8224),                    # five slices of long rows
    (4160, 160), (8192, 2048),      # two row tiles
    (2048, 5632), (2560, 6912),     # ... with three slices, a quad to a wave and for some a second one
    (8256, 288), (16448, 128),      # four, of 16 and 8 waves
    (16448, 4096),                  # four quads to a wave: split in front for four requests
])
def test_rows_of_floats(exe, rows, cols, batch):
    q, x, stride = q4.make(rows, cols, batch, rows + cols + batch)
    x[batch // 2, ::3] = 0.0
    got = q4.run(exe, f"rowsin_{rows}_{cols}_{batch}", q, x, batch, rows, cols, stride)
    q4.check(got, q, x, batch, rows, cols, stride)


def test_one_call_reads_its_rows_only(exe):
    """What lies behind the last row and the last column is not read into the products: infinities there change nothing."""
    rows, cols, batch = 128, 160, 3
    q, x, stride = q4.make(rows, cols, batch, 1)
    want = q4.run(exe, "rowsin_edge", q, x, batch, rows, cols, stride)
    big = np.full((batch + 2, cols), np.inf, np.float32)
    big[1:-1] = x
    d_in, d_out = exe.allocateScratchBuffer(big.nbytes), exe.allocateScratchBuffer(batch * rows * 4)
    try:
        assert exe.uploadToBuffer(d_in, big)
        assert exe.encodeMatMulQ4_0Batched("rowsin_edge", q, d_in + cols * 4, batch, rows, cols, stride, 1, d_out, sync=True), exe.lastError()
        got = np.empty((batch, rows), np.float32)
        assert exe.downloadFromBuffer(d_out, got)
    finally:
        exe.releaseScratchBuffer(d_in)
        exe.releaseScratchBuffer(d_out)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("batch", [1, 4, 5, 8])
@pytest.mark.parametrize("rows,cols,at", [
    (2048, 2048, 0), (4096, 4096, 0),       # in place
    (2048, 2048, -1024), (2048, 2048, 1024),
    (32768, 512, 0), (32768, 512, -32768),  # more workgroups than run at a time
    (256, 8224, 4096),                      # K slices
])
def test_output_over_the_input(exe, rows, cols, batch, at):
    """The output may lie where the input does: all of it is read first.  `at`: floats from the input's start to the output's."""
    q, x, stride = q4.make(rows, cols, batch, rows + cols + batch)
    start, out = max(0, -at), max(0, at)
    room = np.full(max(start + batch * cols, out + batch * rows), np.nan, np.float32)
    room[start:start + batch * cols] = x.reshape(-1)
    dev = exe.allocateScratchBuffer(room.nbytes)
    try:
        for _ in range(3):
            assert exe.uploadToBuffer(dev, room)
            assert exe.encodeMatMulQ4_0Batched(f"over_{rows}_{cols}_{batch}", q, dev + start * 4, batch, rows, cols, stride, 1, dev + out * 4,
                                               sync=True), exe.lastError()
            after = np.empty_like(room)
            assert exe.downloadFromBuffer(dev, after)
            q4.check(after[out:out + batch * rows].reshape(batch, rows), q, x, batch, rows, cols, stride)
    finally:
        exe.releaseScratchBuffer(dev)


@pytest.mark.parametrize("batch", [2, 7])
def test_blocks_far_apart(exe, batch):
    """Every block has a power of two of its own: one whose elements are 2^-60 of another's keeps its 22 bits.  (The large
    ones' weights are zeros: one power of two for a row would leave nothing of what is summed up.)"""
    rows, cols = 256, 512
    q, x, stride = q4.make(rows, cols, batch, 5)
    q.reshape(rows, cols // 32, 18)[:, :8, :2] = 0          # (their scales)
    x[:, :256] *= 2.0 ** 60
    x[0, 32:64] = 0.0
    got = q4.run(exe, f"rowsin_far_{batch}", q, x, batch, rows, cols, stride)
    q4.check(got, q, x, batch, rows, cols, stride)
    x[0, 100] = np.inf
    got = q4.run(exe, f"rowsin_far_{batch}", q, x, batch, rows, cols, stride)
    assert not np.isfinite(got[0]).any() and np.isfinite(got[1:]).all()


@pytest.mark.parametrize("batch", [2, 7])
@pytest.mark.parametrize("exponent", [-88, -100, -118, -130])
def test_tiny_numbers(exe, batch, exponent):
    """The power of two is at most 2^100: smaller elements than 2^-86 have what an fp16 number of theirs has, down to its last
    bit, 2^-24, of which rounding leaves half."""
    rows, cols = 256, 512
    q, x, stride = q4.make(rows, cols, batch, 6)
    x = (x * 2.0 ** exponent).astype(np.float32)
    got = q4.run(exe, f"rowsin_tiny_{batch}", q, x, batch, rows, cols, stride)
    w, x64 = q4.dequant(q, cols), x.astype(np.float64)
    # (2^-149 per addition: sums that are denormal numbers themselves)
    bound = 4e-6 * (np.abs(x64) @ np.abs(w).T) + 2.0 ** -125 * np.abs(w).sum(1) + cols * 2.0 ** -149
    assert (np.abs(got - x64 @ w.T) <= bound).all()
