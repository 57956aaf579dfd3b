"""Q4_0 matmuls whose workgroups outnumber the CUs run on 8 waves instead of 16, two to a CU: plain and with
the SiLU epilogue, at one workgroup more than there are CUs (257 of 64 rows) against one fewer."""
import numpy as np
import pytest

import test_matmul_silu_fusion_gpu as silu
import test_q4_matmul_gpu as q4
from oracle import paged_oracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [255 * 64, 257 * 64])
@pytest.mark.parametrize("cols,batch", [(64, 1), (96, 9), (288, 17), (1056, 32)])
def test_plain(exe, rows, cols, batch):
    q, x, stride = q4.make(rows, cols, batch, rows + cols + batch)
    q4.check(q4.run(exe, f"two_{rows}_{cols}", q, x, batch, rows, cols, stride), q, x, batch, rows, cols, stride)


@pytest.mark.parametrize("form", ["down", "alone"])
@pytest.mark.parametrize("B,hid", [(1, 64), (16, 288), (31, 544)])
def test_silu_epilogue(exe, B, hid, form):
    c = silu.Case(B, hid, 257 * 32, 128, seed=B)
    plain, _ = silu._run(exe, c, form, fuse=0)
    fused, n = silu._run(exe, c, form, fuse=1)
    assert n[0] == 1
    for name in ("gate_up", "gate", "up", "prod"):
        assert np.array_equal(plain[name].view(np.uint8), fused[name].view(np.uint8)), name
    want = po.matmul_q4_0_batched(c.w_gu, c.x, B, 2 * c.ffn, hid)
    assert np.abs(fused["gate_up"] - want).max() <= 2e-5 * np.abs(want).max()
    if form == "down":
        want = po.matmul_q4_0_batched(c.w_down, fused["prod"], B, c.rows_out, c.ffn)
        assert np.abs(fused["down"] - want).max() <= 2e-5 * np.abs(want).max()
