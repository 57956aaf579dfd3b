"""Q4_0 matmuls of long rows: rounding errors grow with the number of blocks a wave adds up in a row, so sums of long
rows are kept in two levels."""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4

pytestmark = pytest.mark.gpu


def _error(exe, rows, cols, batch):
    """2-norm error against float64 of 512 rows (weights and activations spread like normal variables)."""
    rng = np.random.default_rng(rows + cols + batch)
    q = rng.integers(0, 256, (rows, cols // 32, 18), dtype=np.uint8)
    q[:, :, :2] = (0.008 + 0.003 * rng.random((rows, cols // 32, 1))).astype(np.float16).view(np.uint8)
    q = q.reshape(rows, -1)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    got = q4.run(exe, f"long_{rows}_{cols}_{batch}", q, x, batch, rows, cols, q.shape[1])
    pick = np.sort(rng.choice(rows, 512, replace=False))
    want = x.astype(np.float64) @ q4.dequant(q[pick], cols).T
    return np.linalg.norm(got[:, pick] - want) / np.linalg.norm(want)


@pytest.mark.parametrize("rows,cols,batch", [
    (257 * 64, 14336, 2),     # more workgroups than CUs: 8 waves
    (8256, 14336, 17),        # ... because of a second group of requests
    (512, 12256, 3),          # just not split over K: 24 blocks for each of 16 waves
    (512, 11008, 33),
])
def test_error_does_not_grow_with_the_row(exe, rows, cols, batch):
    # 4096 columns are 8 blocks for each of 16 waves.  Sums of one level: 1.22 times that error at 24 blocks in a row and
    # 1.55 times at 56; of two levels: 1.17 times at 56 and less below.
    error, short = _error(exe, rows, cols, batch), _error(exe, 512, 4096, batch)
    print(f"  {rows} x {cols}, {batch} requests: {error:.3e}, 512 x 4096: {short:.3e}", flush=True)
    assert error <= 1.2 * short
