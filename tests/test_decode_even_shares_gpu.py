"""Small launches of the tile-balanced decode kernel whose pairs are whole numbers of a workgroup's least share of tiles:
the ranges end where the pairs end.  Next to them pairs that are not."""
import numpy as np
import pytest

from paged_cases import DeviceCase, assert_parity, make_case, oracle_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(32, 4, 64), (16, 4, 128)])
@pytest.mark.parametrize("tiles", [[10], [10, 12], [0, 10, 14], [10, 11], [48, 52], [9], [10, 0, 30, 4], [160]])
def test_even_shares(exe, tiles, heads, kv_heads, head_dim):
    rows = 64 if head_dim == 64 else 32
    lens = np.array([t * rows - (3 * i + 1 if t else 0) for i, t in enumerate(tiles)])
    case = make_case(f"even.{'.'.join(map(str, tiles))}.{head_dim}", len(tiles), heads, kv_heads, head_dim, 64, lens, seed=len(tiles) + head_dim)
    dev = DeviceCase(exe, case)
    try:
        assert_parity(dev.run(sync=True), oracle_decode(case), 64, case.name)
    finally:
        dev.free()
