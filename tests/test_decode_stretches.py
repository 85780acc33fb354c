"""The decode attention kernel at the edges of its tiles, pages and stretches."""
import pytest
import torch

from aurora_amd import ops
from aurora_amd.ops import torch_ref
from aurora_amd.ops.sequence import Segment, biased_attention

pytestmark = pytest.mark.gpu

#: contexts: tiles of 32, rounds of 128, several stretches
EDGES = [1, 31, 32, 33, 127, 128, 129, 1000, 255, 256, 257, 3001, 5]


def _case(contexts, P, H, G, D, dtype, DV=None, room=0, seed=0):
    g = torch.Generator().manual_seed(seed)
    pages = [-(-c // P) for c in contexts]
    order = torch.randperm(sum(pages) + 1, generator=g)
    bt = torch.zeros(len(contexts), max(max(pages), room // P), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = order[at:at + n]
        at += n
    k, v = (torch.randn(sum(pages) + 1, H // G, P, d, generator=g).to(dtype)
            for d in (D, DV or D))
    q = (torch.randn(len(contexts), H, D, generator=g) * 2).bfloat16()
    return [t.cuda() for t in (q, k, v, bt, torch.tensor(contexts, dtype=torch.int32))]


def _reference(q, k, v, bt, ctx, scale):
    """In 64 bits from the same inputs."""
    P, group = k.shape[2], q.shape[1] // k.shape[1]
    out = torch.zeros(*q.shape[:2], v.shape[3], dtype=torch.float64, device=q.device)
    for s, c in enumerate(ctx.tolist()):
        pages = bt[s, :-(-c // P)].long()
        keys, values = (x.float().double()[pages].transpose(1, 2).reshape(-1, x.shape[1], x.shape[3])
                        [:c].repeat_interleave(group, 1) for x in (k, v))
        w = torch.softmax((keys * q[s].double()).sum(-1) * scale, 0)
        out[s] = (w[:, :, None] * values).sum(0)
    return out


def _check(got, want):
    """Results are those in 64 bits, rounded to bf16: scores of fp32 sums of D products of
    bf16 numbers and weights of 32 bits add less than 2^-12 to the errors of that
    rounding, which moves some of them to the other neighbour: twice that."""
    def errors(x):
        return (x.double() - want).norm(dim=-1) / want.norm(dim=-1)
    assert torch.isfinite(got).all()
    assert (errors(got) <= errors(want.bfloat16()) + 2 ** -11).all()


@pytest.mark.parametrize("P", [16, 48, 64, 256])
@pytest.mark.parametrize("H,G,D", [(8, 4, 128), (4, 2, 64), (7, 7, 128), (2, 1, 64), (20, 20, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("copies", [1, 20])
def test_edges(P, H, G, D, dtype, copies):
    """One copy of the contexts is cut into stretches, twenty of 2 heads or more are not."""
    contexts = EDGES * copies
    args = _case(contexts, P, H, G, D, dtype)
    _check(ops.paged_attention_decode(*args, D ** -0.5), _reference(*args, D ** -0.5))


@pytest.mark.parametrize("window,chunk", [(1, 0), (31, 0), (130, 0), (700, 0), (0, 1), (0, 48),
                                          (0, 500), (0, 0)])
@pytest.mark.parametrize("bias", ["sink", "linear", "log"])
@pytest.mark.parametrize("D,DV", [(64, 128), (128, 64)])
def test_windows(window, chunk, bias, D, DV):
    """Stretches that begin within a tile, and one term more of the denominator."""
    H, G, P = 6, 3, 64
    q, k, v, bt, ctx = _case(EDGES, P, H, G, D, torch.bfloat16, DV, room=8192)
    heads = torch.linspace(0.01, 0.5, H, device="cuda")
    kinds = {"sink": {"slopes": None, "sink": torch.linspace(-3, 3, H, device="cuda")},
             "linear": {"slopes": heads}, "log": {"slopes": heads, "log_rate": heads * 2}}
    out = torch.zeros(len(EDGES), H * DV, device="cuda", dtype=torch.bfloat16)
    seg = Segment(rows=slice(0, len(EDGES)), block_tables=bt, context_lens=ctx, starts=ctx - 1,
                  state_slots=None)
    kind = {"slopes": None, "log_rate": None, "sink": None, **kinds[bias]}
    biased_attention(q, k, v, seg, D ** -0.5, window, kind["slopes"], out, 0, DV, 1.0,
                     kind["log_rate"], kind["sink"], chunk)
    want = torch.zeros(len(EDGES), H * DV)
    on_cpu = [None if t is None else t.cpu() for t in kind.values()]
    torch_ref.biased_attention_paged(
        q.cpu().float(), k.cpu().float(), v.cpu().float(), bt.cpu(),
        torch.arange(len(EDGES) + 1), ctx.cpu(), D ** -0.5, window, on_cpu[0], want, 0, DV, 1.0,
        on_cpu[1], on_cpu[2], chunk)
    _check(out.cpu().view(-1, H, DV), want.double().view(-1, H, DV))


@torch.inference_mode()  # as the engine captures: the generator is shared
def test_replay():
    """The stretches of a captured launch follow the contexts of each replay."""
    H, G, D, P = 8, 4, 128, 64
    q, k, v, bt, ctx = _case(EDGES, P, H, G, D, torch.bfloat16)
    ops.paged_attention_decode(q, k, v, bt, ctx, D ** -0.5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.paged_attention_decode(q, k, v, bt, ctx, D ** -0.5)
    full = ctx.clone()
    for part in (1, 2, 7, 1):
        ctx.copy_((full // part).clamp(min=1))
        graph.replay()
        want = ops.paged_attention_decode(q, k, v, bt, ctx, D ** -0.5)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        _check(got, _reference(q, k, v, bt, ctx, D ** -0.5))
