"""Small launches of the tile-balanced decode kernel leave workgroups without tiles, so that a pair is summed up from fewer
partials: the average tiles per pair at which a workgroup's least share changes, with equal and with mixed lengths (an
empty request among them), both arithmetic modes and more requests than the kernel keeps in registers."""
import numpy as np
import pytest

from paged_cases import DeviceCase, assert_parity, make_case, oracle_decode

pytestmark = pytest.mark.gpu

CUS = 256   # (two workgroups to a CU)


@pytest.mark.parametrize("ratio", [1, 8])
@pytest.mark.parametrize("batch", [1, 3, 66])
@pytest.mark.parametrize("tiles", [1, 2, 3, 8, 9, 47, 48, 159, 160])
def test_least_share(exe, tiles, batch, ratio):
    if batch * tiles > 1500:
        pytest.skip("more tiles than the rule looks at")
    n = tiles * 64
    lens = np.full(batch, n)
    if batch > 1:   # (their average stays)
        lens[0], lens[1] = 0, n + 64 * (tiles // 2)
        lens[-1] -= 64 * (tiles // 2)
    lens = np.maximum(lens - 5, 0)
    case = make_case(f"least.{tiles}.{batch}.{ratio}", batch, ratio, 1, 64, 64, lens, seed=tiles + batch)
    dev = DeviceCase(exe, case)
    try:
        assert_parity(dev.run(sync=True), oracle_decode(case), 64, case.name)
        total, share = max(batch - 1, 1) * tiles, 1 + (tiles == 2 or tiles > 8) + 2 * (tiles >= 48) + 4 * (tiles >= 160)
        assert exe.lastDecodeWorkItems() == min(-(-total // share), CUS * 2)
    finally:
        dev.free()
