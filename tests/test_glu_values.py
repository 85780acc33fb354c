"""The activation behind the products of routed experts and of prompts, value by value."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu

INF = float("inf")


def _products(T, F, W, gates, ups):
    """Rows and weights whose gates and ups are products of two bf16 numbers, which fp32
    holds exactly: gate[t, n] = a[t] c[n], up[t, n] = b[t] d[n]."""
    g = torch.Generator().manual_seed(T + F)
    a, b = (torch.empty(T).uniform_(*s, generator=g).bfloat16() for s in (gates, ups))
    c, d = (torch.empty(F).uniform_(0.5, 1, generator=g).bfloat16() for _ in range(2))
    x, w = torch.zeros(T, W).bfloat16(), torch.zeros(2 * F, W).bfloat16()
    x[:, 0], x[:, 1], w[:F, 0], w[F:, 1] = a, b, c, d
    return x.cuda(), w.cuda()


def _activations(x, w, kernel, limit, alpha, shift, down=None):
    F = w.shape[0] // 2
    if kernel == "prompt":
        from aurora_amd import _hip_ops
        return _hip_ops.many_rows(x, w, True)
    down = torch.eye(x.shape[1], F) if down is None else down  # gives what it reads
    down = down.bfloat16().cuda()
    sel = torch.zeros(x.shape[0], 1, dtype=torch.int32, device="cuda")
    from aurora_amd import _hip_ops
    w, down = w[None].contiguous(), down[None].contiguous()
    y, place = _hip_ops.moe_silu_glu(x, sel, w, down) if kernel == "silu experts" else \
        _hip_ops.moe_clamped_glu(x, sel, w, down, limit, alpha, shift)
    return y[place[:, 0].long(), :F]


#: rows, outputs, width: the tiles of 32, 64, 128 and 256 rows of the experts' kernel, the
#: kernel of any size, prompts
SIZES = [("experts", 40, 192, 192), ("experts", 90, 192, 192), ("experts", 200, 192, 192),
         ("experts", 2100, 1536, 3072), ("experts", 40, 72, 72), ("prompt", 300, 320, 64),
         ("silu experts", 40, 192, 192), ("silu experts", 2100, 1536, 3072)]


@pytest.mark.parametrize("kernel,T,F,W", SIZES)
@pytest.mark.parametrize("limit,alpha,shift", [(INF, 1.0, 0.0), (7.0, 1.702, 1.0)])
def test_rounded_once(kernel, T, F, W, limit, alpha, shift):
    """Results are bf16 roundings of fp32 numbers that a handful of correctly rounded
    operations keep within 2^-21 of the exact value. Where the gate is scaled first, by
    alpha or by log2 e where silu_mul stood before, the exponential multiplies that
    product's and the factor's rounding, 2^-24 each, by its argument."""
    if kernel in ("prompt", "silu experts") and limit < INF:
        pytest.skip("of experts with a limit")
    x, w = _products(T, F, W, (-85.0 / alpha, 20.0), (-9.0, 9.0))
    got = _activations(x, w, kernel, limit, alpha, shift)
    y = x.double() @ w.double().t()
    g, u = y[:, :F].clamp(max=limit), y[:, F:].clamp(-limit, limit) + shift
    z = torch.tensor(alpha, dtype=torch.float32).double().item() * g  # as the kernel has it
    want = g * torch.sigmoid(z) * u
    scaled = 2 if kernel in ("prompt", "silu experts") else alpha != 1
    slack = 2.0 ** -21 + scaled * z.abs() * 2.0 ** -24
    lo, hi = ((want * (1 + s * slack)).float().bfloat16() for s in (-1, 1))
    assert ((got == lo) | (got == hi)).all()


@pytest.mark.parametrize("kernel,T,F,W", SIZES + [("few", 40, 192, 64)])
@pytest.mark.parametrize("limit", [INF, 7.0])
def test_special_values(kernel, T, F, W, limit):
    """NaN stays NaN with and without a limit, a closed gate gives 0 beside any finite
    number, infinities act as in the formula."""
    if kernel in ("prompt", "few", "silu experts") and limit < INF:
        pytest.skip("of experts with a limit")
    x, w = torch.zeros(T, W).bfloat16().cuda(), torch.zeros(2 * F, W).bfloat16().cuda()
    x[:, :2] = 1
    nan = float("nan")
    for a, b in [(nan, 1), (1, nan), (-2e4, 3e38), (-3e38, 3e38), (3, 2), (3e38, 2), (INF, 1),
                 (3, INF), (3, -INF), (-INF, 1), (0, INF)]:
        w[:F, 0], w[F:, 1] = a, b
        if kernel == "few":
            got = ops.linear_silu_mul(x, w).double()
        else:  # the second product adds them up: a row of unlike ones would be NaN
            got = _activations(x, w, kernel, limit, 1.0, 0.0,
                               down=torch.ones(W, F)).double() / (1 if kernel == "prompt" else F)
        g, u = (torch.tensor(v, dtype=torch.float64) for v in (a, b))
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        want = (g / (1 + torch.exp(-g)) * u).float().double().item()
        if want != want:
            assert got.isnan().all(), (a, b)
        elif abs(want) == INF:
            assert (got == want).all(), (a, b)
        else:  # rounded to bf16 twice at most
            assert ((got - want).abs() <= abs(want) * 2 ** -7).all(), (a, b)
