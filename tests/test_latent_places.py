"""Where the visible context of prompt portions lies, against the same in Python."""
import pytest
import torch

from aurora_amd.ops import Segment
from aurora_amd.ops.sequence import _hip

pytestmark = pytest.mark.gpu


#: (context, new tokens) of portions: pages just full, one token, more sequences than a wave
@pytest.mark.parametrize("portions", [[(1, 1)], [(64, 64), (65, 1), (300, 37)],
                                      [(256 + i, 1 + i % 7) for i in range(300)]])
@pytest.mark.parametrize("window", [0, 1, 50])
def test_places(portions, window):
    P, S = 64, len(portions)
    pages = [-(-c // P) for c, _ in portions]
    width = max(pages)
    order = torch.randperm(sum(pages) + 3, generator=torch.Generator().manual_seed(S)).tolist()
    tables = [[order.pop() for _ in range(n)] + [0] * (width - n) for n in pages]
    cu = [0]
    for _, n in portions:
        cu.append(cu[-1] + n)
    ctx = [c for c, _ in portions]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    seg = Segment(rows=slice(0, cu[-1]), block_tables=i32(tables), context_lens=i32(ctx),
                  starts=i32([c - n for c, n in portions]), state_slots=None, cu=i32(cu),
                  cu_host=cu, ctx_host=ctx)
    cache = torch.randn(sum(pages) + 3, 1, P, 8, device="cuda").bfloat16()
    rows, table = seg.latent_rows(cache, window)
    want, n = [], 0
    for s, (c, new) in enumerate(portions):
        lo = max(0, c - new - window + 1) if window else 0
        want += [cache[tables[s][t // P], 0, t % P] for t in range(lo, c)]
        assert table[s].tolist() == [0] * lo + list(range(n, n + c - lo)) + \
            [0] * (table.shape[1] - c)
        n += c - lo
    assert table.shape == (S, max(ctx)) and torch.equal(rows, torch.stack(want))


def test_contexts_beyond_their_pages_are_refused():
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    with pytest.raises(RuntimeError):
        _hip("latent_places").latent_places(i32([[0]]), i32([0, 65]), i32([65]), 64, 0, 65, 65)
