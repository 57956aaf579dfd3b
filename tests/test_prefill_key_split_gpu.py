"""Prefill of few rows: the keys are cut into parts that are added up afterwards.  Against the CPU oracle at
the edges of that rule (15 / 16 key tiles, uneven and empty parts, parts that start inside a group of 64
pages), with the tolerance of test_paged_prefill_gpu.py."""
import numpy as np
import pytest

from mlcompiler_amd.workloads import make_prefill
from test_paged_prefill_gpu import check, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,D,P,chunk,ctx", [
    (8, 1, 64, 64, 32, [448]), (8, 1, 64, 64, 32, [449]),   # 15 and 16 tiles
    (8, 1, 128, 32, 19, [4500, 3]),      # 142 pages of one tile; nearly all parts of one request are empty
    (4, 1, 128, 64, 70, [600, 0, 1111]), # GQA ratio 4, several row blocks, a request without a prefix
    (4, 2, 64, 128, 33, [2000]), (2, 2, 128, 64, 5, [3001]),
    (16, 2, 64, 32, 77, [700, 90, 1300]),
    (8, 1, 64, 64, 600, [0]),            # causal from scratch: the first rows see one part only
])
def test_prefill_parts(exe, H, Hkv, D, P, chunk, ctx):
    w = make_prefill(len(ctx), chunk, H, Hkv, D, P, ctx, seed=H + D + chunk)
    _, got, _ = check(exe, w, "parts")
    assert np.array_equal(got, run_gpu(exe, w, sync=False))
