"""Reductions over a row's lanes: the row's largest magnitude and its sum of squares, whichever lane holds what matters."""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4
from oracle import paged_oracle as po
from test_matmul_norm_fusion_gpu import EPS, _pool, _read

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [16, 70])           # a row per workgroup, four rows per workgroup
def test_the_largest_element_in_every_lane(exe, batch):
    """One element of a row is 2^20 times the others, in another column for every row: its scale is the row's."""
    rows, cols = 64, 2048
    q, x, stride = q4.make(rows, cols, batch, batch)
    w = q4.dequant(q, cols)
    for turn in range(3):
        v = x.copy()
        at = (np.arange(batch) * 131 + turn * 677) % cols
        v[np.arange(batch), at] = 2.0 ** 20
        got = q4.run(exe, f"lanes_{batch}", q, v, batch, rows, cols, stride)
        assert (np.abs(got - v.astype(np.float64) @ w.T) <= 4e-6 * (np.abs(v.astype(np.float64)) @ np.abs(w).T)).all()


@pytest.mark.parametrize("n", [8, 512, 520, 4096, 8200])
def test_norms_of_rows_with_one_element(exe, n):
    """A row with one element that is not zero has the norm sqrt(n) there, whichever lane holds it."""
    rows = 96
    x = np.zeros((rows, n), np.float32)
    at = (np.arange(rows) * 89) % n
    x[np.arange(rows), at] = 3.0
    gamma = np.linspace(0.5, 1.5, n).astype(np.float32)[: n - 3]      # (1 beyond)
    d_x, d_y = _pool(exe, x), _pool(exe, np.full_like(x, np.nan))
    try:
        for fuse in (0, 1):
            assert exe.setOption("fuse_row_ops", fuse)
            assert exe.beginForwardPassCB() and exe.encodeRmsNormBatched(d_x, gamma, EPS, rows, n, d_y) and exe.flushForwardPassCB()
            got = _read(exe, d_y, x)
            want = po.rms_norm_batched(x, gamma, EPS, rows, n)
            assert np.abs(got - want).max() <= 2e-6 * np.abs(want).max()
    finally:
        exe.setOption("fuse_row_ops", 1)
        for b in (d_x, d_y):
            exe.releaseScratchBuffer(b)
