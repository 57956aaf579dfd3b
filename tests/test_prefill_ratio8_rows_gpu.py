"""GQA ratio 8 with as many workgroups as leave the keys in one part: 32 rows of eight heads per workgroup up to a number of
key tiles and where blocks of 64 rows would take another round over the CUs, else 64 rows of four heads."""
import pytest

from mlcompiler_amd.workloads import make_prefill
from test_paged_prefill_gpu import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,tiles", [(64, 9), (64, 10), (128, 15), (128, 16)])
@pytest.mark.parametrize("chunk,page", [(129, 64), (150, 32), (192, 64)])     # a row, a part and all of the last 64 rows
def test_on_both_sides_of_the_rule(exe, D, tiles, chunk, page):
    longest = tiles * 32 - chunk        # (the row block that sees the most ends with a tile, or in it)
    w = make_prefill(3, chunk, 72, 9, D, page, [longest, 0, longest - 31], seed=tiles + chunk)
    check(exe, w, f"{tiles} tiles")


@pytest.mark.parametrize("D", [64, 128])
def test_one_kv_head(exe, D):
    w = make_prefill(2, 2500, 8, 1, D, 128, [3, 70], seed=D)      # 2 x 79 row blocks of 32
    check(exe, w, "one KV head")


@pytest.mark.parametrize("chunk,batch", [(5, 128), (5, 129), (33, 129), (70, 64), (70, 65)])    # (twice 128 and four times 64: all CUs once)
def test_on_both_sides_of_a_round(exe, chunk, batch):
    w = make_prefill(batch, chunk, 8, 1, 64, 64, [320 - chunk - r % 50 for r in range(batch)], seed=batch)
    check(exe, w, f"{batch} of {chunk}")
