"""The encoder's kernels at the edges of their tiles, over strided rows, and short rows of
the norms."""
import itertools

import pytest
import torch

from aurora_amd import ops
from aurora_amd.ops import torch_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H,G", [(64, 12, 12), (128, 4, 2), (64, 6, 2)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("scale", [None, -0.3, 0.0])
def test_attention_edges(D, H, G, causal, scale):
    lens = [1, 31, 32, 33, 63, 64, 65, 0, 127, 128, 129, 256, 300, 2]
    scale = D ** -0.5 if scale is None else scale
    g = torch.Generator(device="cuda").manual_seed(D + H)
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    rows = torch.randn(sum(lens), H + 2 * G, D, generator=g, device="cuda").bfloat16()
    rows[:, H:H + G] *= 3  # sharp weights, and references that move
    q, k, v = rows.split([H, G, G], 1)
    got = ops.attention_prefill(q, k, v, cu, scale, causal).double()
    assert torch.equal(got, ops.attention_prefill(
        q.contiguous(), k.contiguous(), v.contiguous(), cu, scale, causal).double())
    for a, b in zip(cu.tolist(), cu.tolist()[1:]):
        if a == b:
            continue
        kk, vv = (t[a:b].double().repeat_interleave(H // G, 1).transpose(0, 1) for t in (k, v))
        w = q[a:b].double().transpose(0, 1) @ kk.transpose(1, 2) * scale
        if causal:
            w = w.masked_fill(torch.ones(b - a, b - a, device="cuda").triu(1).bool(),
                              float("-inf"))
        want = (torch.softmax(w, -1) @ vv).transpose(0, 1)
        err = (got[a:b] - want).norm(dim=-1) / want.norm(dim=-1)
        # weights are good to 2^-22, results are rounded once to 2^-9 of themselves
        assert err.max() < 2 ** -8, (b - a, float(err.max()))


@pytest.mark.parametrize("D,H,G", [(64, 3, 1), (128, 2, 2), (20, 3, 3)])
def test_rotation_in_place_of_strided_rows(D, H, G):
    x = torch.randn(37, H + 2 * G, D, device="cuda").bfloat16()
    pos = torch.randint(0, 90, (37,), device="cuda", dtype=torch.int32)
    cs = torch_ref.rope_cos_sin_cache(D, 90, 1e4).cuda()
    want = torch_ref.rope_apply(x[:, :H].cpu(), x[:, H:H + G].cpu(), pos.cpu(), cs.cpu())
    rest = x[:, H + G:].clone()
    ops.rope_apply_(x[:, :H], x[:, H:H + G], pos, cs)
    assert torch.equal(x[:, H + G:], rest)
    for a, b in zip((x[:, :H], x[:, H:H + G]), want):  # at most one rounding the other way
        assert (a.cpu().float() - b.float()).abs().max() <= 2 ** -8 * b.float().abs().max()


@pytest.mark.parametrize("scale", [0.125, -0.1])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D,H,G", [(64, 4, 2), (128, 2, 2)])
def test_attention_rotates_as_the_rotation_does(D, H, G, causal, scale):
    lens = [1, 31, 63, 64, 65, 127, 128, 129, 0, 200, 300]  # tiles of 64 keys, 128 rows
    cu = torch.tensor([0, *itertools.accumulate(lens)], dtype=torch.int32, device="cuda")
    x = torch.randn(sum(lens), H + 2 * G, D, device="cuda").bfloat16()
    pos = torch.cat([torch.arange(n) for n in lens]).int().cuda()
    cs = torch_ref.rope_cos_sin_cache(D, max(lens), 1e4).cuda()
    q, k, v = x.split([H, G, G], dim=1)
    before = x.clone()
    got = ops.attention_prefill_turned(q, k, v, cs, cu, scale, causal)
    assert torch.equal(x, before)
    q, k = ops.rope_apply(q.clone(), k.clone(), pos, cs)
    want = ops.attention_prefill(q, k, v, cu, scale, causal)
    # a rotated number may be rounded the other way, by 2^-8 of itself: scores of D of them
    # move by some 2^-8 of their spread of scale sqrt(D)
    err = (got.float() - want.float()).norm(dim=(1, 2)) / want.float().norm(dim=(1, 2))
    assert err.max() < 2 ** -7, float(err.max())


@pytest.mark.parametrize("T,H", [(1, 8), (5, 64), (4, 504), (3, 512), (7, 520), (9, 768),
                                 (2, 1016), (6, 1024), (3, 1032)])
def test_short_rows_of_the_norms(T, H):
    x, r = (torch.randn(T, H, device="cuda").bfloat16() for _ in range(2))
    w = (1 + 0.1 * torch.randn(H, device="cuda")).bfloat16()

    def close(a, b):  # fp32 inside, rounded once or twice to 2^-9
        return (a.double().cpu() - b.double()).abs().max() <= 2 ** -7 * b.double().abs().max()

    unit = lambda y: y / (y.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()  # noqa: E731
    assert close(ops.rmsnorm(x, w, 1e-5), (unit(x.double()) * w.double()).cpu())
    got, total = ops.rmsnorm_residual(x, r, w, 1e-5)
    both = x.double() + r.double()
    assert torch.equal(total, both.float().bfloat16())
    assert close(got, (unit(both) * w.double()).cpu())


@pytest.mark.parametrize("H", [8, 64, 100, 768, 1000, 2048])
def test_pool(H):
    lens = [1, 2, 9, 10, 11, 130, 300]
    cu = torch.tensor([0] + lens).cumsum(0).int()
    h = torch.randn(sum(lens), H, device="cuda").bfloat16()
    got = ops.embed_pool(h, cu.cuda()).double().cpu()
    for s, (a, b) in enumerate(zip(cu.tolist(), cu.tolist()[1:])):
        want = h[a:b].double().mean(0).cpu()
        want = want / want.norm()
        assert (got[s] - want).norm() < 2 ** -8  # rounded once to 2^-9
