"""Routers of few tokens, whose logits come in parts, on both sides of the rule for them."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 17, 128, 129])
@pytest.mark.parametrize("W,E,top", [(4096, 8, 2), (3712, 8, 8), (1792, 31, 3), (2048, 64, 64),
                                     (320, 512, 70), (256, 300, 9), (200, 400, 5)])
def test_choices_and_weights(T, W, E, top):
    """Whole logits, exact in fp32 in any order, so that choices are the reference's, equal
    ones too; then random ones."""
    g = torch.Generator().manual_seed(W + E)
    h, router = (torch.randint(0, 2, (n, W), generator=g).bfloat16() * 2 - 1 for n in (T, E))
    bias = torch.randperm(E, generator=g).float() * 2
    logits = h.double() @ router.double().t() + bias.double()
    sel, gate = ops._hip.moe_route(h.cuda(), router.cuda(), bias.cuda(), top)
    want = logits.sort(dim=1, descending=True, stable=True)
    assert torch.equal(sel.cpu().long(), want.indices[:, :top])
    assert torch.allclose(gate.cpu().double(), want.values[:, :top].softmax(1), rtol=1e-5,
                          atol=1e-12)
    for corr in (torch.randn(E, generator=g), None):
        _compare(g, T, W, E, top, 1, 1, corr)


def _compare(g, T, W, E, top, groups, keep, corr):
    """Random logits against 64 bits: the same experts wherever the last one and the last group
    are chosen by more than 1e-4, which is more than any order of summing moves them."""
    h, router = (torch.randn(n, W, generator=g).bfloat16() for n in (T, E))
    router = (router * 2 * W ** -0.5).contiguous()
    z = h.double() @ router.double().t()
    score = z.softmax(1) if corr is None else z.sigmoid()
    choice = z if corr is None else score + corr.double()
    of = choice.view(T, groups, -1)
    of = of.amax(2) if corr is None or E == groups else of.topk(2, 2).values.sum(2)
    order = of.sort(dim=1, descending=True)
    choice = choice.view(T, groups, -1).masked_fill(
        (torch.zeros(T, groups).scatter(1, order.indices[:, :keep], 1.0) == 0)[:, :, None],
        -torch.inf).view(T, E)
    best = choice.sort(dim=1, descending=True)
    clear = torch.ones(T, dtype=torch.bool)
    if keep < groups:
        clear &= order.values[:, keep - 1] - order.values[:, keep] > 1e-4
    if top < E:
        clear &= best.values[:, top - 1] - best.values[:, top] > 1e-4
    assert clear.float().mean() > 0.9 or T == 1
    at = best.indices[:, :top]
    want = torch.zeros(T, E).double().scatter(1, at, score.gather(1, at))
    if corr is not None:
        want /= want.sum(1, keepdim=True) + 1e-20
    sel, gate = ops._hip.moe_route_grouped(
        h.cuda(), router.cuda(), None if corr is None else corr.cuda(), top, groups, keep, 2.5)
    got = torch.zeros(T, E).scatter(1, sel.cpu().long(), gate.cpu())
    assert torch.equal((got > 0)[clear], (want > 0)[clear])
    assert torch.allclose(got[clear].double(), 2.5 * want[clear], rtol=1e-4, atol=1e-7)


GROUPED = [(2048, 64, 8, 3, 6), (512, 512, 64, 5, 8), (512, 512, 512, 9, 7), (2560, 96, 3, 2, 64),
           (7168, 256, 8, 4, 8), (4096, 130, 13, 13, 70)]


@pytest.mark.parametrize("T", [1, 17, 128, 129])
@pytest.mark.parametrize("W,E,groups,keep,top", GROUPED)
@pytest.mark.parametrize("sigmoid", [False, True])
def test_groups(T, W, E, groups, keep, top, sigmoid):
    g = torch.Generator().manual_seed(W + E + T)
    _compare(g, T, W, E, top, groups, keep, torch.randn(E, generator=g) if sigmoid else None)


@pytest.mark.parametrize("W,E,groups,keep,top", GROUPED + [
    (4096, 8, 1, 1, 2), (3712, 8, 1, 1, 8), (1792, 31, 1, 1, 3), (2880, 32, 1, 1, 4),
    (256, 300, 1, 1, 9), (320, 512, 1, 1, 70)])
def test_as_among_many(W, E, groups, keep, top):
    """A token's experts and weights are the same, to the last bit, whatever tokens are beside
    it: few of them come in parts, 300 of them do not."""
    g = torch.Generator(device="cuda").manual_seed(W + E)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda")  # noqa: E731
    h, router, bias = rnd(300, W).bfloat16(), (rnd(E, W) * 2 * W ** -0.5).bfloat16(), rnd(E)
    for route in (lambda x: ops._hip.moe_route(x, router, bias, top),
                  lambda x: ops._hip.moe_route(x, router, None, top),
                  lambda x: ops._hip.moe_route_grouped(x, router, bias, top, groups, keep, 2.5),
                  lambda x: ops._hip.moe_route_grouped(x, router, None, top, groups, keep, 2.5)):
        sel, gate = route(h)
        for a, b in ((0, 1), (3, 20), (20, 52), (52, 85), (172, 300)):
            s, w = route(h[a:b])
            assert torch.equal(s, sel[a:b]) and torch.equal(w, gate[a:b])
