"""Norms of rows that a workgroup holds and of rows that it reads twice."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [1032, 2040, 2048, 2056, 4096, 4104, 8184, 8192, 8200, 16400])
@pytest.mark.parametrize("parts", [0, 1, 2, 4, 5, 9])
@pytest.mark.parametrize("T", [1, 3])
def test_against_64_bits(T, H, parts):
    """Around the widths that one, two and four vectors a thread hold. The stream's new rows
    are what is added up in fp32 and rounded; of the norm 2^-8 is two roundings to bf16."""
    g = torch.Generator().manual_seed(H + parts)
    x = torch.randn(max(parts, 1), T, H, generator=g)
    res, w = torch.randn(T, H, generator=g).bfloat16(), torch.randn(H, generator=g).bfloat16()
    # one part is a plain product
    x = x[0].bfloat16() if parts <= 1 else x
    total = x if parts <= 1 else sum(x).bfloat16()  # in fp32, one after the other
    want = (total.float() + res.float()).bfloat16()
    h, new = ops.rmsnorm_residual(x.cuda(), res.cuda(), w.cuda(), 1e-5)
    exact = total.double() + res.double()
    norm = want.double() * torch.rsqrt(exact.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    assert torch.equal(new.cpu(), want)
    assert (h.cpu().double() - norm).abs().le(norm.abs() * 2 ** -8 + 1e-6).all()
    plain = ops.rmsnorm(want.cuda(), w.cuda(), 1e-5).cpu().double()
    norm = want.double() * torch.rsqrt(want.double().pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    assert (plain - norm).abs().le(norm.abs() * 2 ** -8 + 1e-6).all()
