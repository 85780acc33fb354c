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


def _activations(x, w, kernel, limit, alpha, shift):
    F = w.shape[0] // 2
    if kernel == "prompt":
        from aurora_amd import _hip_ops
        return _hip_ops.many_rows(x, w, True)
    eye = torch.eye(x.shape[1], F).bfloat16().cuda()  # what the second product reads
    sel = torch.zeros(x.shape[0], 1, dtype=torch.int32, device="cuda")
    from aurora_amd import _hip_ops
    y, place = _hip_ops.moe_clamped_glu(x, sel, w[None].contiguous(), eye[None].contiguous(),
                                        limit, alpha, shift)
    return y[place[:, 0].long(), :F]


#: rows, outputs, width: the tiles of 32, 64, 128 and 256 rows of the experts' kernel, the
#: kernel of any size, prompts
SIZES = [("experts", 40, 192, 192), ("experts", 90, 192, 192), ("experts", 200, 192, 192),
         ("experts", 2100, 1536, 3072), ("experts", 40, 72, 72), ("prompt", 300, 320, 64)]


@pytest.mark.parametrize("kernel,T,F,W", SIZES)
@pytest.mark.parametrize("limit,alpha,shift", [(INF, 1.0, 0.0), (7.0, 1.702, 1.0)])
def test_rounded_once(kernel, T, F, W, limit, alpha, shift):
    """Results are bf16 roundings of fp32 numbers that a handful of correctly rounded
    operations keep within 2^-21 of the exact value; where the gate is scaled first, the
    exponential multiplies that rounding by its argument."""
    if kernel == "prompt" and limit < INF:
        pytest.skip("prompts have no limit")
    x, w = _products(T, F, W, (-85.0 / alpha, 20.0), (-9.0, 9.0))
    got = _activations(x, w, kernel, limit, alpha, shift)
    y = x.double() @ w.double().t()
    g, u = y[:, :F].clamp(max=limit), y[:, F:].clamp(-limit, limit) + shift
    z = torch.tensor(alpha, dtype=torch.float32).double().item() * g  # as the kernel has it
    want = g * torch.sigmoid(z) * u
    slack = 2.0 ** -21 + (alpha != 1) * z.abs() * 2.0 ** -24
    lo, hi = ((want * (1 + s * slack)).float().bfloat16() for s in (-1, 1))
    assert ((got == lo) | (got == hi)).all()
