"""Products of few rows and many outputs in float32: the bits of the bf16 ones."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 17, 32, 33, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("N,K", [(n, k) for n in (8256, 16387, 40001) for k in (64, 2048, 4160)]
                         + [(48, 128), (516, 64)])
def test_bits(M, N, K):
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = torch.randn(N, K, device="cuda").bfloat16()
    x[0, 0] = float("inf")
    mine = ops._hip.own_product(x, w, 3) is not None
    assert mine == (M <= 64 and (N * K * 2 >> 20 <= 128 or M <= 32 and K < 4096))
    y = ops.linear_float(x, w)
    assert y.dtype == torch.float32
    assert torch.equal(y.view(torch.int32), ops.linear(x, w).float().view(torch.int32))
    wide = torch.randn(M, 2 * K, device="cuda").bfloat16()[:, K:]  # strided rows
    assert torch.equal(ops.linear_float(wide, w), ops.linear(wide, w).float())


def test_forms_that_are_not_taken():
    """Few outputs (K in parts), many rows, other types: the product and a conversion."""
    for m, n, k, dtype in ((3, 512, 8192, torch.bfloat16), (300, 9000, 512, torch.bfloat16),
                           (4, 9000, 100, torch.bfloat16), (4, 9000, 512, torch.float32)):
        x, w = (torch.randn(*s, device="cuda").to(dtype) for s in ((m, k), (n, k)))
        y = ops.linear_float(x, w)
        assert y.dtype == torch.float32 and torch.equal(y, ops.linear(x, w).float())
