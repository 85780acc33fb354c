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


@pytest.mark.parametrize("T,W,times", [(257, 1024, 4), (257, 1028, 4), (257, 2048, 4),
                                       (257, 4096, 4), (3, 2048, 16), (3, 4096, 4), (3, 8192, 4)])
@pytest.mark.parametrize("kind", ["delta", "gate", "moe", "post", "convolution"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_of_the_residual(T, W, times, kind, dtype):
    """The same of the residual's norm: rows with zeros behind them go through LDS. What is
    normed before it is added has a weight that takes the larger factor back."""
    g = torch.Generator(device="cuda").manual_seed(W + T)

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    x, w, step, factor = rnd(T, W), rnd(W), rnd(W), times ** 0.5
    kw = {"delta": rnd(T, W).to(dtype), "step": step}
    if kind == "gate":
        kw["gate"] = rnd(T, W).to(dtype), rnd(W)
    if kind == "moe":
        place = torch.randperm(3 * T, generator=g, device="cuda").view(T, 3).int()
        kw["moe"] = rnd(3 * T, W).to(dtype), place, torch.rand(T, 3, generator=g, device="cuda")
    if kind == "post":
        kw["post"] = rnd(W)
    ring, taps = rnd(T, 4, W).to(dtype), rnd(5, W)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    seg = ops.Segment(slice(0, T), i32(0)[None], i32(1), torch.arange(T, device="cuda").int() * 3,
                      torch.arange(T, device="cuda").int() - 1)

    def run(n, k):
        def wide(t):
            if isinstance(t, tuple):
                return tuple(v if v.dtype == torch.int32 or v.shape[-1] != W else wide(v)
                             for v in t)
            return pad(t, (0, n))

        on = {name: wide(v) for name, v in kw.items()}
        if "post" in on:
            on["post"] = on["post"] / k
        xs, past = wide(x), wide(ring * k)
        if kind == "convolution":
            out = ops.residual_rmsnorm_conv(xs, wide(w), EPS / k ** 2, wide(taps), past, [seg],
                                            dtype=dtype, **on)
        else:
            out = ops.residual_rmsnorm(xs, wide(w), EPS / k ** 2, dtype=dtype, **on),
        return [xs, *(t / k for t in (*out, past))]

    for a, b in zip(run(0, 1.0), run(W * (times - 1), factor)):
        assert torch.equal(a, b[..., :W])
