"""Q6_K matmul: one, two and four row tiles per workgroup, incomplete last workgroups, batches at the edges of the
accumulators in use, rows with fewer groups than waves and with a last round that is not full."""
import numpy as np
import pytest

from test_q6k_matmul_gpu import check, make, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [
    (32, 256), (96, 2304),       # one tile per workgroup; four of eight waves have a group, the last round is half full
    (257 * 32, 256),             # two, one tile behind the last workgroup's
    (1003 * 32, 256),            # four (up to 32 requests), three tiles in the last workgroup
])
@pytest.mark.parametrize("batch", [1, 8, 9, 16, 17, 32, 33, 64])
def test_tiles(exe, rows, cols, batch):
    q, x, stride = make(rows, cols, batch, rows + batch)
    check(run(exe, f"tiles.{rows}.{cols}.{batch}", q, x, batch, rows, cols, stride), q, x, batch, rows, cols, stride)
