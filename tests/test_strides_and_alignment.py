"""Rows and heads in every layout that counts as contiguous, at every address."""
import pytest
import torch

from aurora_amd import ops
from aurora_amd.ops import torch_ref

pytestmark = pytest.mark.gpu


def _one_head(T, D, g):
    """[T, 1, D] of one head, cut from heads that lie one after another: contiguous, though
    the stride of its heads is T D."""
    x = torch.randn(1, T, D, generator=g).bfloat16().cuda().transpose(0, 1)
    assert x.is_contiguous() and (T == 1 or x.stride(1) != D)
    return x


def _off(t, elements=1):
    """The same at an address off by some elements."""
    flat = torch.empty(t.numel() + elements, dtype=t.dtype, device="cuda")
    out = flat[elements:].view(t.shape)
    return out.copy_(t)


@pytest.mark.parametrize("T", [1, 2, 9])
def test_rotation_of_one_head(T):
    g = torch.Generator().manual_seed(T)
    q, k = _one_head(T, 64, g), _one_head(T, 64, g)
    cs = torch_ref.rope_cos_sin_cache(64, 32, 10000.0, dtype=torch.float32)
    at = torch.arange(T, dtype=torch.int32)
    want = torch_ref.rope_apply(q.cpu().float(), k.cpu().float(), at, cs)
    got = ops.rope_apply(q, k, at.cuda(), cs.cuda())
    for a, b in zip(got, want):
        assert ((a.cpu().float() - b).abs() <= b.abs() * 2 ** -8 + 2 ** -12).all()


@pytest.mark.parametrize("H,G,D", [(4, 2, 64), (1, 1, 128), (3, 1, 64)])
@pytest.mark.parametrize("layout", ["off", "one head"])
@pytest.mark.parametrize("lens", [[1], [5, 70, 33]])
def test_packed_attention(H, G, D, layout, lens):
    if layout == "one head" and (H, G) != (1, 1):
        pytest.skip("of one head")
    g = torch.Generator().manual_seed(D)
    cu = torch.tensor([0] + lens).cumsum(0).int()
    T = int(cu[-1])
    if layout == "off":
        q, k, v = (_off(torch.randn(T, h, D, generator=g).bfloat16()) for h in (H, G, G))
    else:
        q, k, v = (_one_head(T, D, g) for _ in range(3))
    got = ops.attention_prefill(q, k, v, cu.cuda(), D ** -0.5, causal=False)
    want = torch_ref.attention_prefill(q.cpu().float(), k.cpu().float(), v.cpu().float(), cu,
                                       D ** -0.5, False)
    assert (got.cpu().float() - want).norm() <= 2 ** -7.5 * want.norm()


def test_packed_attention_of_a_longer_buffer():
    """Keys and values may have rows past the queries' last."""
    q, k, v = (torch.randn(n, 2, 64, device="cuda").bfloat16() for n in (40, 64, 50))
    cu = torch.tensor([0, 15, 40], dtype=torch.int32, device="cuda")
    got = ops.attention_prefill(q, k, v, cu, 0.125, causal=True)
    assert torch.equal(got, ops.attention_prefill(q, k[:40], v[:40], cu, 0.125, causal=True))


@pytest.mark.parametrize("P", [16, 64])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("elements", [1, 3, 4])
def test_prompts_over_a_cache_at_an_odd_address(P, cache, elements):
    g = torch.Generator().manual_seed(P)
    D, L, n = 64, 150, 40
    k, v = (_off(torch.randn(-(-L // P), 2, P, D, generator=g).to(cache), elements)
            for _ in range(2))
    q = torch.randn(n, 4, D, generator=g).bfloat16()
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32)  # noqa: E731
    args = torch.arange(-(-L // P), dtype=torch.int32)[None], i32(0, n), i32(L)
    got = ops.attention_prefill_paged(q.cuda(), k, v, *(a.cuda() for a in args), D ** -0.5)
    want = ops.attention_prefill_paged(q.cuda(), k.clone(), v.clone(),
                                       *(a.cuda() for a in args), D ** -0.5)
    assert torch.equal(got, want)


@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("P", [16, 64])
def test_prompts_beside_rows_without_keys(P, cache):
    """Rows whose context says that there are none read nothing and disturb nobody."""
    g = torch.Generator().manual_seed(P)
    n = -(-40 // P)
    k, v = (torch.randn(n, 1, P, 64, generator=g).to(cache).cuda() for _ in range(2))
    q = torch.randn(80, 4, 64, generator=g).bfloat16().cuda()
    bt = torch.arange(n, dtype=torch.int32, device="cuda").expand(2, n).contiguous()
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    got = ops.attention_prefill_paged(q, k, v, bt, i32(0, 40, 80), i32(40, 0), 0.125)
    want = ops.attention_prefill_paged(q[:40], k, v, bt[:1], i32(0, 40), i32(40), 0.125)
    assert torch.equal(got[:40], want)


def test_experts_of_rows_at_an_odd_address():
    from aurora_amd.models.config import get_spec
    from aurora_amd.models.llama import MoEMLP
    m = MoEMLP(get_spec("smoke-moe"), torch.bfloat16).cuda()
    for p in m.parameters():
        p.data.normal_(0, p.shape[-1] ** -0.5)
    x = torch.randn(300, 512, device="cuda").bfloat16()
    got, want = m(_off(x)), m(x)
    assert (got.float() - want.float()).norm() <= 2 ** -6 * want.float().norm()
