"""Products without rows, outputs or terms."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(0, 128, 4096), (1, 0, 64), (7, 0, 4096), (33, 0, 2048),
                                   (100, 0, 8192), (300, 0, 768), (5, 128, 0), (200, 64, 0)])
def test_empty(m, n, k):
    x = torch.ones(m, k, dtype=torch.bfloat16, device="cuda")
    w = torch.ones(n, k, dtype=torch.bfloat16, device="cuda")
    for got in (ops.linear(x, w), ops.linear_parts(x, w)):
        assert got.shape == (m, n) and got.dtype == torch.bfloat16 and not got.any()
    if n:
        silu = ops.linear_silu_mul(x, w)
        assert silu.shape == (m, n // 2) and not silu.any()
