"""Products on both sides of the lines between the kernels and the library."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


def _inputs(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w = (torch.randn(r, k, generator=g, device="cuda") for r in (m, n))
    return x.bfloat16(), (w * k ** -0.5).bfloat16()


def _close(got, want):
    assert got.dtype == torch.bfloat16 and got.shape == want.shape
    # a rounding of the result and, unless they are fused, of what is activated
    assert (got.double() - want).norm() <= 2 ** -7.5 * want.norm()


@pytest.mark.parametrize("m,n,k", [
    (32, 16448, 4096), (33, 16448, 4096), (32, 16448, 4160), (64, 256, 192),  # 128 MB
    (65, 2048, 3072), (65, 3072, 3072), (96, 2048, 8192), (96, 1984, 8192), (128, 8192, 3072),
    (128, 8256, 3072), (128, 64, 14336), (129, 64, 14336),
    (191, 5120, 2112), (192, 5120, 2112), (256, 6144, 4096), (256, 6208, 4096),
    (256, 5120, 2048), (257, 5120, 2112)])
def test_plain(m, n, k):
    x, w = _inputs(m, n, k)
    want = x.double() @ w.double().t()
    _close(ops.linear(x, w), want)
    parts = ops.linear_parts(x, w)
    _close(parts if parts.dim() == 2 else parts.sum(0).bfloat16(), want)


@pytest.mark.parametrize("m,n,k", [
    (32, 64, 3072), (32, 64, 3136), (32, 2816, 4096), (32, 2784, 4096), (32, 5120, 5120),
    (64, 1024, 2048), (64, 992, 2048), (64, 5120, 4096), (64, 8224, 4096), (64, 13120, 4096),
    (96, 1792, 2048), (96, 1760, 2048), (96, 8192, 4096), (128, 5120, 2048), (128, 5088, 2048),
    (128, 64, 1024), (128, 64, 1088), (255, 6144, 768), (256, 6144, 768), (700, 4096, 1536),
    (500, 8192, 1536), (1000, 3072, 2112), (1030, 3072, 2112), (2048, 3072, 2112),
    (2600, 1280, 2112)])
def test_silu(m, n, k):
    x, w = _inputs(m, 2 * n, k)
    y = x.double() @ w.double().t()
    _close(ops.linear_silu_mul(x, w), torch.nn.functional.silu(y[:, :n]) * y[:, n:])
