"""Routed silu GLU experts of plain decoders through the grouped kernels."""
import pytest
import torch

from aurora_amd import ops
from aurora_amd.models.config import ModelSpec
from aurora_amd.models.llama import MoEMLP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 15, 16, 17, 130, 700])
@pytest.mark.parametrize("W,F,E,top", [(64, 64, 4, 1), (128, 192, 8, 2), (448, 320, 3, 3)])
def test_against_every_expert_by_itself(T, W, F, E, top):
    g = torch.Generator(device="cuda").manual_seed(T + W)
    n = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, router = n(T, W).bfloat16(), (n(E, W) * W ** -0.5).bfloat16()
    gu, dn = (n(E, 2 * F, W) * W ** -0.5).bfloat16(), (n(E, W, F) * F ** -0.5).bfloat16()
    got = ops.moe_silu_glu(x, router, top, gu, dn).double()
    z = (x.double() @ router.double().t()).bfloat16().double()
    best = z.topk(min(top + 1, E), -1).values
    # where the choice hangs on the last bit of a logit either is right
    clear = torch.ones(T, dtype=torch.bool, device="cuda") if top == E else \
        best[:, top - 1] - best[:, top] > 0.02
    val, sel = z.topk(top, -1)
    w = val.softmax(-1)
    want = torch.zeros_like(got)
    for e in range(E):
        a, b = (x.double() @ gu[e].double().t()).chunk(2, -1)
        y = (torch.nn.functional.silu(a) * b) @ dn[e].double().t()
        want += y * (w * (sel == e)).sum(-1, keepdim=True)
    err = ((got - want).norm(dim=-1) / want.norm(dim=-1))[clear]
    # logits, activations, rows and results are each rounded to 2^-9 of themselves
    assert clear.any() and err.max() < 2 ** -6


def test_experts_share_one_tensor_and_follow_a_move():
    spec = ModelSpec(name="m", hidden_size=64, n_layers=1, n_heads=1, n_kv_heads=1, head_dim=64,
                     intermediate_size=64, vocab_size=8, n_experts=4)
    moe = MoEMLP(spec, torch.bfloat16)
    for p in moe.parameters():
        p.data.normal_(0, 0.1)
    moe = moe.cuda()
    x = torch.randn(9, 64, device="cuda").bfloat16()
    first = moe(x)
    assert moe.experts[3].down.weight.data_ptr() == moe._w_dn[3].data_ptr()
    moe.experts[0].down.weight.data.zero_()  # seen by the next pass
    moe.experts[1].down.weight.data.zero_()
    moe.experts[2].down.weight.data.zero_()
    moe.experts[3].down.weight.data.zero_()
    assert first.abs().max() > 0 and moe(x).abs().max() == 0
