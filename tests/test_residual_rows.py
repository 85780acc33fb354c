"""Norms of the fp32 residual: rows that threads hold and rows in LDS, deltas whole and in parts."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [4, 1022, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196])
@pytest.mark.parametrize("T", [3, 257])
@pytest.mark.parametrize("kind", ["none", "delta", "parts2", "parts9", "gate", "moe", "post"])
def test_against_64_bits(T, W, kind):
    """Around the widths that one and two vectors a thread hold, of few rows and of many. A
    delta in parts is their sum in fp32, rounded; the residual is off by some 2^-24 of what
    was added, the norm by a rounding to bf16 besides: half a unit of 8 bits, up to 2^-8 of
    the value."""
    g = torch.Generator().manual_seed(W + T)

    def rnd(*shape):
        return torch.randn(*shape, generator=g)

    x, w, step, kw = rnd(T, W), rnd(W), None, {}
    delta = rnd(T, W).bfloat16()
    if kind != "none":
        kw["delta"], step = delta, rnd(W)
    if kind.startswith("parts"):
        kw["delta"] = rnd(int(kind[5:]), T, W)
        delta = sum(kw["delta"]).bfloat16()  # in fp32, one after the other
    d = delta.double() if kind != "none" else torch.zeros(T, W).double()
    size = x.double().abs() + d.abs() + 1
    if kind == "gate":
        kw["gate"] = rnd(T, W + 12).bfloat16()[:, :W], rnd(W)
        d = d * torch.sigmoid(kw["gate"][0].double() + kw["gate"][1].double())
    if kind == "moe":
        rows, place = rnd(3 * T, W).bfloat16(), torch.randperm(3 * T, generator=g).view(T, 3)
        kw["moe"] = rows, place.int(), torch.rand(T, 3, generator=g)
        terms = rows.double()[place] * kw["moe"][2].double().unsqueeze(-1)
        d, size = d + terms.sum(1), size + terms.abs().sum(1)
    if kind == "post":
        kw["post"] = rnd(W)
        d = d * torch.rsqrt(d.pow(2).mean(-1, keepdim=True) + 1e-5) * kw["post"].double()
        size += d.abs()
    if step is not None:
        kw["step"], d, size = step, d + step.double(), size + step.double().abs()
    new = x.double() + d
    want = new * torch.rsqrt(new.pow(2).mean(-1, keepdim=True) + 1e-5) * (1 + w.double())
    xg = x.cuda()
    on = {k: tuple(t.cuda() for t in v) if isinstance(v, tuple) else v.cuda()
          for k, v in kw.items()}
    got = ops.residual_rmsnorm(xg, w.cuda(), 1e-5, dtype=torch.bfloat16, **on)
    # 16 steps of 2^-24 for the sums, the sigmoid and the factor of the norm
    assert (xg.cpu().double() - new).abs().le(size * 2 ** -20).all()
    assert (got.cpu().double() - want).abs().le(
        want.abs() * 2 ** -8 + size * (1 + w.double().abs()) * 2 ** -19).all()


@pytest.mark.parametrize("W", [288, 1028, 4100])
def test_parts_before_a_convolution(W):
    """Single tokens: the same bits as of the parts' sum, held by threads or in LDS."""
    from test_sequence_kernels import _segment, _to
    seg = _to(_segment([1] * 4, [37, 7, 116, 1], 64, [4, 0, 2, 5], True)[0], "cuda")
    parts, x = torch.randn(3, 4, W, device="cuda"), torch.randn(4, W, device="cuda")
    w, taps = torch.randn(W, device="cuda"), torch.randn(4, W, device="cuda")
    ring = torch.randn(6, 3, W, device="cuda").bfloat16()
    out = []
    for delta in (parts, (parts[0] + parts[1] + parts[2]).bfloat16()):
        xs, past = x.clone(), ring.clone()
        out.append((*ops.residual_rmsnorm_conv(xs, w, 1e-5, taps, past, [seg], delta=delta,
                                               dtype=torch.bfloat16), xs, past))
    for a, b in zip(*out):
        assert torch.equal(a, b)
