"""A batch that does not fill its tile of 32 requests: the Q4_0 and Q6_K kernels read nobody else's activation
fragments (tolerance: see test_matmul_tokens_gpu.py)."""
import numpy as np
import pytest

import test_q4_matmul_gpu as q4
import test_q6k_matmul_gpu as q6
from oracle import paged_oracle as po
from test_matmul_tokens_gpu import check

pytestmark = pytest.mark.gpu

@pytest.mark.parametrize("batch", [1, 8, 9, 16, 17, 31, 33, 63])
def test_small_batch_does_not_read_other_requests(exe, batch):
    # the fragments of a full batch of infinities lie in the workspace behind this batch's own
    rows, cols = 256, 512
    q, x, stride = q4.make(rows, cols, 64, 3)
    q4.run(exe, "tok_few", q, np.full_like(x, np.inf), 64, rows, cols, stride)
    check(q4.run(exe, "tok_few", q, x[:batch], batch, rows, cols, stride), q4.dequant(q, cols), x[:batch])
    q, x, stride = q6.make(rows, cols, 64, 3)
    q6.run(exe, "tok_few6", q, np.full_like(x, np.inf), 64, rows, cols, stride)
    check(q6.run(exe, "tok_few6", q, x[:batch], batch, rows, cols, stride), po.dequantize_q6_k(q, cols), x[:batch])
