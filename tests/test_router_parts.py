"""Routers of few tokens, whose logits come in parts, on both sides of the rule for them."""
import pytest
import torch

from aurora_amd import ops
from aurora_amd.ops import torch_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 17, 128, 129])
@pytest.mark.parametrize("W,E,top", [(4096, 8, 2), (3712, 8, 8), (1792, 31, 3), (2048, 64, 64),
                                     (320, 512, 70), (256, 300, 9), (200, 400, 5)])
def test_choices_and_weights(T, W, E, top):
    """Whole logits, exact in fp32 in any order, so that choices are the reference's, equal
    ones too; then random ones, off by less than 1e-4 in whatever order they are summed."""
    g = torch.Generator().manual_seed(W + E)
    h, router = (torch.randint(0, 2, (n, W), generator=g).bfloat16() * 2 - 1 for n in (T, E))
    bias = torch.randperm(E, generator=g).float() * 2
    logits = h.double() @ router.double().t() + bias.double()
    sel, gate = ops._hip.moe_route(h.cuda(), router.cuda(), bias.cuda(), top)
    want = logits.sort(dim=1, descending=True, stable=True)
    assert torch.equal(sel.cpu().long(), want.indices[:, :top])
    assert torch.allclose(gate.cpu().double(), want.values[:, :top].softmax(1), rtol=1e-5,
                          atol=1e-12)
    h, router = (torch.randn(n, W, generator=g).bfloat16() for n in (T, E))
    router = (router * 2 * W ** -0.5).contiguous()
    for corr in (torch.randn(E, generator=g), None):
        if corr is None:
            s, w = torch_ref.moe_route_softmax(h, router, top, 1, 1, 2.5)
        else:
            s, w = torch_ref.moe_route_grouped(h, router, corr, top, 1, 1, 2.5)
        sel, gate = ops._hip.moe_route_grouped(
            h.cuda(), router.cuda(), None if corr is None else corr.cuda(), top, 1, 1, 2.5)
        scores = torch.zeros(T, E).scatter(1, s.long(), w)
        got = torch.zeros(T, E).scatter(1, sel.cpu().long(), gate.cpu())
        # the last chosen may change places with one as good, once
        assert ((got > 0) == (scores > 0)).float().mean() > 1 - 2 / E / T
        both = (got > 0) & (scores > 0)
        assert torch.allclose(got[both], scores[both], rtol=1e-4, atol=1e-7)
