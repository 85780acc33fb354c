"""The norm of a single row in the product that reads it."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,S", [(64, 16), (192, 3), (1024, 2), (1088, 8), (2048, 7), (2112, 2),
                                 (4096, 4), (4160, 2), (8192, 2)])
@pytest.mark.parametrize("N", [16, 48, 4112])
@pytest.mark.parametrize("silu", [False, True])
def test_against_64_bits(K, S, N, silu):
    """Around the widths that one to eight vectors a thread hold and fewer steps of K than are
    asked for ahead. The normed row is rounded to bf16 (2^-8), so is the result."""
    g = torch.Generator().manual_seed(K + N + S)
    parts = torch.randn(S, 1, K, generator=g)
    res, w = torch.randn(1, K, generator=g).bfloat16(), torch.randn(K, generator=g).bfloat16()
    wt = (torch.randn(N * (1 + silu), K, generator=g) * K ** -0.5).bfloat16()
    new = torch.empty(1, K, dtype=torch.bfloat16, device="cuda")
    y = ops._hip.one_row_product(parts.cuda(), res.cuda(), w.cuda(), 1e-5, new, wt.cuda(), silu)
    total = sum(parts).bfloat16().float() + res.float()  # in fp32, one after the other
    assert torch.equal(new.cpu(), total.bfloat16())
    inv = torch.rsqrt(total.double().pow(2).mean() + 1e-5)
    h = total.bfloat16().double() * inv * w.double()
    z, off = h @ wt.double().t(), (h.abs() @ wt.double().abs().t()) * 2 ** -8 + 1e-6
    if silu:
        gate, up = z.split(N, 1)
        # silu's slope is at most 1.1
        z = torch.nn.functional.silu(gate) * up
        off = off[:, :N] * 1.1 * (up.abs() + off[:, N:]) + off[:, N:] * gate.abs()
    got = (y.sum(0) if y.dim() == 3 else y).cpu().double()
    assert (got - z).abs().le(off + z.abs() * 2 ** -8 + 1e-6).all()


@pytest.mark.parametrize("K,S", [(64, 16), (192, 3), (576, 5), (1024, 16), (1088, 8), (1984, 2),
                                 (2048, 7), (2112, 2), (4096, 4), (4160, 2), (8192, 2)])
@pytest.mark.parametrize("silu", [False, True])
def test_bits_of_the_separate_norm(K, S, silu):
    """64 rows, as a last bit of the sum of squares seldom shows in bf16."""
    N = 4112
    g = torch.Generator(device="cuda").manual_seed(K + S)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda")  # noqa: E731
    w, wt = rnd(K).bfloat16(), (rnd(N * (1 + silu), K) * K ** -0.5).bfloat16()
    x, res = rnd(S, 64, K) * rnd(64, K).exp(), (rnd(64, K) * rnd(64, K).exp()).bfloat16()
    for r in range(64):
        row, old = x[:, r:r + 1].contiguous(), res[r:r + 1].clone()
        new = torch.empty_like(old)
        y = ops._hip.one_row_product(row, old, w, 1e-5, new, wt, silu)
        h, want = ops.rmsnorm_residual(row, old, w, 1e-5)
        assert torch.equal(new, want)
        z = ops._hip.silu_few_rows(h, wt) if silu else ops._hip.linear_few_rows(h, wt, True)
        assert torch.equal(y, z)


def test_rows_that_are_normed_before():
    """More rows, whole ones, more parts than a thread holds: as ever."""
    w = torch.randn(4096, device="cuda").bfloat16()
    wt = torch.randn(6144, 4096, device="cuda").bfloat16()
    for x, mine in ((torch.randn(4, 1, 4096), True), (torch.randn(5, 1, 4096), False),
                    (torch.randn(4, 2, 4096), False), (torch.randn(1, 4096).bfloat16(), False)):
        x = x.cuda()
        res = torch.randn(x.shape[-2], 4096, device="cuda").bfloat16()
        rows, new = ops.norm_ahead(x, res, w, 1e-5, wt, False)
        assert isinstance(rows, ops.Unnormed) == mine
        h, want = ops.rmsnorm_residual(x, res, w, 1e-5)
        assert torch.equal(ops.linear_parts(rows, wt), ops.linear_parts(h, wt))
        assert torch.equal(new, want)  # (written by the product)
        assert not isinstance(ops.norm_ahead(x, res, w, 1e-5, None, False)[0], ops.Unnormed)
