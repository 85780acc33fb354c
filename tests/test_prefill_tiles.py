"""The prompt attention kernel at the edges of its tiles, pages and steps."""
import pytest
import torch

from aurora_amd import ops
from aurora_amd.ops import torch_ref

pytestmark = pytest.mark.gpu

#: new and cached tokens of each sequence: one row, steps of 32, tiles of 64, blocks of
#: 64 to 256 rows, each just missed and just met
EDGES = [(1, 0), (1, 63), (2, 62), (31, 0), (32, 1), (33, 95), (63, 0), (64, 64), (65, 127),
         (0, 5), (129, 200), (257, 3), (300, 0)]


def _case(P, H, G, D, dtype, spread=1.0, seed=0):
    g = torch.Generator().manual_seed(seed)
    kv = H // G
    ctx = [n + p for n, p in EDGES]
    pages = [-(-c // P) for c in ctx]
    order = torch.randperm(sum(pages) + 1, generator=g)
    bt = torch.zeros(len(EDGES), max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = order[at:at + n]
        at += n
    k, v = (torch.randn(sum(pages) + 1, kv, P, D, generator=g).to(dtype) for _ in range(2))
    q = (torch.randn(sum(n for n, _ in EDGES), H, D, generator=g) * spread).bfloat16()
    cu = torch.tensor([0] + [n for n, _ in EDGES]).cumsum(0).int()
    return [t.cuda() for t in (q, k, v, bt, cu, torch.tensor(ctx, dtype=torch.int32))]


def _reference(q, k, v, bt, cu, ctx, scale):
    """In 64 bits from the same inputs."""
    P, out = k.shape[2], torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    group = q.shape[1] // k.shape[1]
    for s in range(len(ctx)):
        a, b, c = int(cu[s]), int(cu[s + 1]), int(ctx[s])
        pages = bt[s, :-(-c // P)].long()
        keys, values = (x.float().double()[pages].transpose(1, 2).reshape(-1, x.shape[1], x.shape[3])
                        [:c].repeat_interleave(group, 1) for x in (k, v))
        hidden = torch.arange(c, device=q.device)[None] > \
            torch.arange(c - (b - a), c, device=q.device)[:, None]
        for h in range(q.shape[1]):
            w = (q[a:b, h].double() @ keys[:, h].t()) * scale
            w = torch.softmax(w.masked_fill(hidden, float("-inf")), -1)
            out[a:b, h] = w @ values[:, h]
    return out


@pytest.mark.parametrize("P", [16, 48, 64, 256])
@pytest.mark.parametrize("H,G,D", [(4, 4, 128), (8, 2, 64), (7, 7, 128), (2, 1, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_edges(P, H, G, D, dtype):
    args = _case(P, H, G, D, dtype)
    got = ops.attention_prefill_paged(*args, D ** -0.5).double()
    want = _reference(*args, D ** -0.5)
    # weights and results are rounded to 2^-9 of themselves, the weights' errors average;
    # the largest of a row's results is about its norm over sqrt(D) times 4
    err = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() < 2 ** -7


@pytest.mark.parametrize("scale", [-0.09, 0.0, 0.7])
def test_scales_and_rising_scores(scale):
    """Scores of both signs, none, and ones that rise far past the reference of the
    softmax again and again: weights of 2^-9 stay exact to 2^-7 in all."""
    args = _case(64, 4, 4, 128, torch.bfloat16, spread=3.0, seed=1)
    k, bt, ctx = args[1], args[3], args[5]
    for s in range(len(EDGES)):  # later keys are longer
        for t in range(int(ctx[s])):
            k[int(bt[s, t // 64]), :, t % 64] *= 0.1 + t / 64
    got = ops.attention_prefill_paged(*args, scale).double()
    want = _reference(*args, scale)
    err = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() < 2 ** -6  # a weight near 1 beside another: twice a result's rounding


def test_block_search_over_many_sequences():
    """More sequences than a wave has lanes: blocks find their rows past 64 and 128."""
    n, P, D = 150, 64, 64
    lens = [1 + (i * 37) % 90 for i in range(n)]
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    k, v = (torch.randn(2 * n, 1, P, D, device="cuda").bfloat16() for _ in range(2))
    bt = torch.arange(2 * n, dtype=torch.int32, device="cuda").view(n, 2)
    q = torch.randn(sum(lens), 4, D, device="cuda").bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32, device="cuda")
    got = ops.attention_prefill_paged(q, k, v, bt, cu, ctx, 0.125).float().cpu()
    want = torch_ref.attention_prefill_paged(
        *(t.float().cpu() if t.is_floating_point() else t.cpu()
          for t in (q, k, v, bt, cu, ctx)), 0.125)
    err = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() < 2 ** -7


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.bfloat16),
                                     (128, torch.float8_e4m3fn)])
def test_results_into_a_buffer(D, dtype):
    """Prompts and decoding rows of one batch write their parts of one tensor."""
    q, k, v, bt, cu, ctx = _case(64, 8, 4, D, dtype)
    one = q[:len(ctx)].contiguous()
    want = ops.attention_prefill_paged(q, k, v, bt, cu, ctx, 0.1)
    last = ops.paged_attention_decode(one, k, v, bt, ctx, 0.1)
    both = torch.full((len(q) + len(one) + 1, *q.shape[1:]), 7.0, device="cuda").bfloat16()
    ops.attention_prefill_paged(q, k, v, bt, cu, ctx, 0.1, out=both[:len(q)])
    ops.paged_attention_decode(one, k, v, bt, ctx, 0.1, out=both[len(q):-1])
    assert torch.equal(both[:len(q)], want) and torch.equal(both[len(q):-1], last)
    assert (both[-1] == 7).all()
    for wrong in (both[1:], both[:len(q)].float(), both[:len(q), ::2]):
        with pytest.raises(RuntimeError):
            ops.attention_prefill_paged(q, k, v, bt, cu, ctx, 0.1, out=wrong)
        with pytest.raises(RuntimeError):
            ops.paged_attention_decode(one, k, v, bt, ctx, 0.1, out=wrong)
