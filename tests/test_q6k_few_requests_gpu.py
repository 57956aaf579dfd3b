"""Q6_K matmul around the numbers of requests at which a product holds both parts of the activations (up to 16) or not."""
import pytest

import test_q6k_matmul_gpu as q6

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 4, 5, 7, 8, 9, 15, 16, 17])
@pytest.mark.parametrize("rows,cols", [(32, 256), (96, 512), (8224, 256), (16480, 256)])   # one, two and four row tiles
def test_both_parts_in_one_product(exe, rows, cols, batch):
    q, x, stride = q6.make(rows, cols, batch, rows + batch)
    x[batch // 2, 1::2] = 0.0
    got = q6.run(exe, f"q6few_{rows}_{batch}", q, x, batch, rows, cols, stride)
    q6.check(got, q, x, batch, rows, cols, stride)
