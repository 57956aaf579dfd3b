"""The tile-balanced decode kernel on the matrix pipe away from its full groups and whole-tile pages:
GQA ratios that fill neither the waves nor the sixteen columns, and pages smaller than a tile (each
wave's slice of a tile in a page of its own), with lengths around slice, page and tile boundaries.
Slots behind a request's last token hold NaN, which nothing may read into a product."""
import numpy as np
import pytest

from paged_cases import DeviceCase, assert_parity, make_case, oracle_decode

pytestmark = pytest.mark.gpu

LENS = [1, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 127, 129, 0, 1030, 2100]


@pytest.mark.parametrize("D,P", [(64, 16), (64, 32), (64, 64), (64, 192), (128, 8), (128, 16), (128, 32)])
@pytest.mark.parametrize("ratio", [1, 2, 3, 5, 6, 7, 12, 16])
def test_group_and_page_sizes(exe, D, P, ratio):
    case = make_case(f"r{ratio}_d{D}_p{P}", len(LENS), 2 * ratio, 2, D, P, LENS, seed=ratio * P + D)
    print(f"[case] {case.name}", flush=True)
    for pool in (case.k_pages, case.v_pages):
        rows = pool.view(np.float16).reshape(case.capacity_pages, P, 2 * D)
        used = np.zeros((case.capacity_pages, P), bool)
        for r, n in enumerate(LENS):
            for i in range(n):
                used[case.page_tables_flat[case.page_table_offsets[r] + i // P], i % P] = True
        rows[~used] = np.nan
    dev = DeviceCase(exe, case)
    try:
        got = dev.run()
        assert exe.lastDecodeKernel().startswith(f"stream<{D},"), exe.lastDecodeKernel()
        assert exe.setOption("decode_grid_wgs", 5)      # few workgroups: ranges of many pairs, other cuts
        again = dev.run()
    finally:
        exe.setOption("decode_grid_wgs", 0)
        dev.free()
    want = oracle_decode(case)
    assert_parity(got, want, D, case.name)
    assert_parity(again, want, D, case.name + " (second cut)")
