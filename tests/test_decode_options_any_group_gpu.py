"""The decode options reach the builds for partly filled groups and small pages as well."""
import numpy as np
import pytest

from paged_cases import DeviceCase, assert_parity, make_case, oracle_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [5, 70])               # figures of the requests in registers, in LDS
@pytest.mark.parametrize("D,P,ratio", [(64, 64, 3), (64, 16, 8), (128, 32, 6), (128, 8, 12)])
def test_weights_and_stages_follow_the_options(exe, batch, D, P, ratio):
    lens = np.random.default_rng(ratio).integers(1, 900, batch)
    c = make_case(f"opt_{D}_{P}_{ratio}_{batch}", batch, 2 * ratio, 2, D, P, lens, seed=ratio)
    want = oracle_decode(c)
    dev = DeviceCase(exe, c)
    where = "regs" if batch <= 64 else "lds"
    try:
        default = dev.run()
        assert f"mfma-p32,{where},2>" in exe.lastDecodeKernel()
        assert_parity(default, want, D, c.name)
        assert exe.setOption("decode_pv_fp16", 1)
        half = dev.run()
        assert f"mfma,{where},2>" in exe.lastDecodeKernel()
        assert_parity(half, want, D, c.name + " fp16 weights")
        assert not np.array_equal(half, default)
        e_half, e_full = (np.sqrt(np.mean((x.astype(np.float64) - want) ** 2)) for x in (half, default))
        assert e_half > 8 * e_full                       # (weights of 11 bits instead of 22)
        assert exe.setOption("decode_pv_fp16", 0)
        for stages in (3, 4):
            assert exe.setOption("decode_stages", stages)
            got = dev.run()
            assert f"mfma-p32,{where},{min(stages, 4 if batch <= 64 else 3)}>" in exe.lastDecodeKernel()
            assert_parity(got, want, D, f"{c.name} {stages} stages")
    finally:
        exe.setOption("decode_pv_fp16", 0)
        exe.setOption("decode_stages", 0)
        dev.free()
