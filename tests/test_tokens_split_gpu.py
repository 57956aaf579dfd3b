"""Matmuls over more than 64 tokens: the split of their activations at the widths where its workgroups change (4096
columns) and where a row no longer fits the registers (8192), with the bound of test_matmul_tokens_gpu.py."""
import pytest

from test_matmul_tokens_gpu import check, q4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [65, 131])
@pytest.mark.parametrize("cols", [4064, 4096, 4128, 8160, 8192, 8224])
def test_widths(exe, cols, tokens):
    rows = 64
    q, x, stride = q4.make(rows, cols, tokens, cols + tokens)
    check(q4.run(exe, f"split_{cols}_{tokens}", q, x, tokens, rows, cols, stride), q4.dequant(q, cols), x)
