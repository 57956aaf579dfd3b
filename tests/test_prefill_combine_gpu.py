"""Prefill of few rows: the sum over the parts takes eight of them at a time.  Against the CPU oracle at part
counts around a multiple of eight and at the most there are (two key tiles per part here, up to 64 parts), with the
tolerance of test_paged_prefill_gpu.py; the last block of rows is not full."""
import pytest

from mlcompiler_amd.workloads import make_prefill
from test_paged_prefill_gpu import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,D,chunk", [(8, 1, 64, 5), (8, 1, 128, 33), (2, 2, 64, 70), (8, 2, 128, 3)])
@pytest.mark.parametrize("tiles", [3, 4, 14, 16, 18, 34, 300])
def test_part_counts(exe, tiles, H, Hkv, D, chunk):
    w = make_prefill(2, chunk, H, Hkv, D, 64, [max(0, tiles * 32 - chunk), 40], seed=tiles + D + chunk)
    check(exe, w, f"{tiles} tiles")
