"""Q4_0 matmuls of up to 64 requests at the edges of the kernel's division: 1, 2 or 4 accumulator registers per
product (batches 4 | 5, 8 | 9), groups of 16 requests (one, two or four to a workgroup), incomplete quads of blocks, waves without a quad and with one or
two, 1, 2 or 4 tiles of 16 rows per workgroup, 8 or 16 waves; and a matmul that both finishes one RMSNorm and
carries the residual add of the next (its two norms have weights of their own)."""
import numpy as np
import pytest

import test_decode_split_fusion_gpu as split
import test_matmul_rope_fusion_gpu as rope
import test_matmul_silu_fusion_gpu as silu
import test_q4_matmul_gpu as q4
from oracle import paged_oracle as po
from paged_cases import make_case
from test_matmul_norm_fusion_gpu import EPS, _pool, _read
from test_matmul_tokens_gpu import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 4, 5, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("rows,cols", [
    (64, 64),        # half a quad of blocks, most waves without one
    (4160, 160),     # a quad and one block; two tiles per workgroup, four from 17 requests on (65 row groups)
    (192, 2080),     # 17 quads, the last incomplete: one wave has two
    (8256, 1184),    # wide: four tiles per workgroup, 16 waves (8 from 17 requests on), 10 quads
])
def test_divisions(exe, rows, cols, batch):
    q, x, stride = q4.make(rows, cols, batch, rows + cols + batch)
    got = q4.run(exe, f"groups_{rows}_{cols}_{batch}", q, x, batch, rows, cols, stride)
    check(got, q4.dequant(q, cols), x)
    assert np.array_equal(got, q4.run(exe, f"groups_{rows}_{cols}_{batch}", q, x, batch, rows, cols, stride, sync=False))


@pytest.mark.parametrize("rows,cols,batch", [
    (10240, 160, 17), (10240, 1184, 32),      # two groups of 16 requests in a workgroup, the second with one request and full
    (6144, 2080, 33), (6144, 160, 48), (28672, 96, 31),    # ... the last one missing, two rounds of the CUs
    (10240, 96, 49), (10240, 1184, 64),       # four groups
])
def test_groups_that_share_a_workgroup(exe, rows, cols, batch):
    q, x, stride = q4.make(rows, cols, batch, rows + cols + batch)
    name = f"share_{rows}_{cols}_{batch}"
    got = q4.run(exe, name, q, x, batch, rows, cols, stride)
    check(got, q4.dequant(q, cols), x)
    bad = batch - 17 if batch > 32 else batch - 1
    x[bad] = np.inf                # stays in its row, also where the last quad of blocks is incomplete
    keep = np.arange(batch) != bad
    assert np.array_equal(got[keep], q4.run(exe, name, q, x, batch, rows, cols, stride)[keep])


@pytest.mark.parametrize("rows,cols,batch,ksplit", [
    (64, 96, 3, 0), (192, 2080, 17, 0),                       # one tile and group per workgroup; incomplete quads
    (8256, 160, 5, 0), (10240, 1184, 33, 0),                  # four tiles
    (10240, 160, 17, 0), (10240, 1184, 64, 0), (4160, 96, 100, 0),    # ... and two groups of requests
    (512, 14336, 9, 0), (512, 4096, 21, 3), (192, 2080, 70, 2),       # K slices
])
def test_weights_as_pairs(exe, rows, cols, batch, ksplit):
    q, x, stride = q4.make(rows, cols, batch, rows + cols + batch)
    assert exe.setOption("q4_int_operand", 0) and exe.setOption("q4_ksplit", ksplit)
    try:
        got = q4.run(exe, f"pairs_{rows}_{cols}_{batch}", q, x, batch, rows, cols, stride)
        again = q4.run(exe, f"pairs_{rows}_{cols}_{batch}", q, x, batch, rows, cols, stride, sync=False)
    finally:
        exe.setOption("q4_int_operand", 1)
        exe.setOption("q4_ksplit", 0)
    check(got, q4.dequant(q, cols), x)
    assert np.array_equal(got, again)


@pytest.mark.parametrize("batch", [17, 32, 49, 64])
def test_silu_of_groups_that_share_a_workgroup(exe, batch):
    c = silu.Case(batch, 160, 5120, 192, seed=batch)
    got, n = silu._run(exe, c, "down", fuse=1)
    assert n == (1, 1)
    check(got["gate_up"], q4.dequant(c.w_gu, 160), c.x)
    _, _, want = po.gate_up_split_silu_mul(got["gate_up"], batch, 5120, 10240)
    assert np.max(np.abs(got["prod"] - want) / (np.abs(want) + 1e-30)) < 5e-6      # (as in test_matmul_silu_fusion_gpu.py)
    check(got["down"], q4.dequant(c.w_down, 5120), got["prod"])


@pytest.mark.parametrize("batch", [17, 32, 33, 64])    # four tiles per workgroup of 16 waves, of 8 from 33 requests on
def test_rope_of_four_tiles(exe, batch):
    c = rope.Case(B=batch, H=40, Hkv=4, D=128, hid=1184, seed=batch)
    plain, _ = rope._run(exe, c, "scatter", fuse=0)
    fused, n = rope._run(exe, c, "scatter", fuse=1)
    assert n == 1
    for m in ("qkv", "q", "k", "v", "kp", "vp"):
        assert np.array_equal(plain[m].view(np.uint8), fused[m].view(np.uint8)), m
    check(fused["qkv"], q4.dequant(c.w, c.hid), c.x)
    wants = po.qkv_split_rope_cast(fused["qkv"], c.cos, c.sin, c.B, c.H, c.Hkv, c.D, c.rows, c.q_rows, c.kv_rows, c.kv_rows, c.rotary)
    for m, want in zip("qkv", wants):
        assert np.array_equal(fused[m].view(np.uint8), np.ascontiguousarray(want).view(np.uint8)), m


@pytest.mark.parametrize("batch", [1, 6, 16, 21, 40])
def test_a_chain_of_norms(exe, batch):
    """matmul, add, norm, matmul, add, norm, matmul: the one in the middle finishes the first norm and starts the second."""
    rng = np.random.default_rng(batch)
    n = 512
    w = [po.quantize_q4_0((rng.standard_normal((r, n)) * 0.05).astype(np.float32)) for r in (n, n, 2 * n)]
    gamma = [(1.0 + 0.3 * rng.standard_normal(n)).astype(np.float32) for _ in range(2)]
    x, r0, r1 = (rng.standard_normal((batch, n)).astype(np.float32) for _ in range(3))
    like = {m: np.empty((batch, 2 * n if m == "y" else n), np.float32) for m in ("p0", "h0", "n0", "p1", "h1", "n1", "y")}
    dev = {m: _pool(exe, np.full_like(a, np.nan)) for m, a in like.items()}
    src = [_pool(exe, a) for a in (x, r0, r1)]
    before = exe.fusedMatmulNormLaunches()
    try:
        assert exe.beginForwardPassCB()
        for i, (a, p, r, h, norm) in enumerate(((src[0], "p0", src[1], "h0", "n0"), (dev["n0"], "p1", src[2], "h1", "n1"))):
            assert exe.encodeMatMulQ4_0Batched(f"norms{batch}.{i}", w[i], a, batch, n, n, w[i].shape[1], 1, dev[p])
            assert exe.encodeAddBatched(dev[p], r, dev[h], batch * n)
            assert exe.encodeRmsNormBatched(dev[h], gamma[i], EPS, batch, n, dev[norm])
        assert exe.encodeMatMulQ4_0Batched(f"norms{batch}.2", w[2], dev["n1"], batch, 2 * n, n, w[2].shape[1], 1, dev["y"])
        assert exe.flushForwardPassCB(), exe.lastError()
        got = {m: _read(exe, dev[m], like[m]) for m in like}
    finally:
        for buf in list(dev.values()) + src:
            exe.releaseScratchBuffer(buf)
    assert exe.fusedMatmulNormLaunches() - before == (1 if batch <= 32 else 0) + 1   # (40: the norm has more elements than the reader's threads)
    for a, m, i in ((x, "p0", 0), (got["n0"], "p1", 1), (got["n1"], "y", 2)):
        check(got[m], q4.dequant(w[i], n), a)
    for i, r in enumerate((r0, r1)):
        assert np.array_equal(got[f"h{i}"], r + got[f"p{i}"])
        want = po.rms_norm_batched(got[f"h{i}"], gamma[i], EPS, batch, n)
        # (as in test_matmul_norm_fusion_gpu.py: a sum of n squares and one rounding per factor)
        assert (np.abs(got[f"n{i}"] - want) <= 2e-6 * np.abs(want).max(axis=1, keepdims=True)).all()


@pytest.mark.parametrize("batch", [1, 3, 4, 5, 7, 8, 9])
def test_few_requests_behind_every_producer(exe, batch):
    """The fragments of up to 4, up to 8 and more requests lie differently: written by the decode attention (with a
    request without tokens) and by the SiLU epilogue, behind a matmul whose input the split kernel wrote."""
    rng = np.random.default_rng(batch)
    lens = rng.integers(1, 300, batch)
    lens[batch // 2] = 0
    case = make_case(f"few.{batch}", batch, 16, 2, 64, 64, lens, seed=batch)
    w = po.quantize_q4_0((rng.standard_normal((192, 1024)) * 0.05).astype(np.float32))
    o, out, _, n, _ = split._run(exe, case, w, 192, "proj", fuse=1)
    assert n == 1
    check(out, q4.dequant(w, 1024), o.reshape(batch, 1024))
    c = silu.Case(batch, 160, 4128, 192, seed=batch)
    got, n = silu._run(exe, c, "down", fuse=1)
    assert n == (1, 1)
    check(got["gate_up"], q4.dequant(c.w_gu, 160), c.x)
    check(got["down"], q4.dequant(c.w_down, 4128), got["prod"])
