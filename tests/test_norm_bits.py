"""Norms of rows that threads hold give the bits of the kernels that read a row twice."""
import pytest
import torch
from torch.nn.functional import pad

from aurora_amd import ops

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -17


@pytest.mark.parametrize("H,times", [(1032, 16), (2048, 16), (2888, 4), (4096, 4), (8192, 4)])
@pytest.mark.parametrize("parts", [0, 3])
def test_of_the_stream(H, times, parts):
    """Rows with zeros behind them, too long to be held: every thread adds the same squares in
    the same order, the mean and eps are a power of four smaller and the factor a power of two
    larger, all exactly. 4096 rows, as a last bit of the sum seldom shows in bf16."""
    g = torch.Generator(device="cuda").manual_seed(H)

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    T, wide = 64 if parts else 4096, (0, H * (times - 1))
    for _ in range(8 if parts else 1):
        x = rnd(parts, T, H) if parts else (rnd(T, H) * rnd(T, H).exp()).bfloat16()
        res, w = (rnd(T, H) * rnd(T, H).exp()).bfloat16(), rnd(H).bfloat16()
        h, new = ops.rmsnorm_residual(x, res, w, EPS)
        want, stream = ops.rmsnorm_residual(pad(x, wide), pad(res, wide), pad(w, wide),
                                            EPS / times)
        assert torch.equal(new, stream[:, :H])
        assert torch.equal(h * times ** 0.5, want[:, :H])
