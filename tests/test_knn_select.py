"""Nearest documents: shares of workgroups, selection among equal scores, special values."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


def _unit(n, d, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.nn.functional.normalize(torch.randn(n, d, generator=g), dim=-1).cuda()


#: documents: fewer than neighbours, tiles of 16, shares of 128, more than one list a thread
@pytest.mark.parametrize("n", [1, 15, 17, 63, 64, 65, 127, 129, 1000, 5000, 66000, 600000])
@pytest.mark.parametrize("q,k", [(1, 1), (1, 20), (3, 64), (16, 40), (8, 17)])
@pytest.mark.parametrize("dtype,d", [(torch.float32, 64), (torch.bfloat16, 128),
                                     (torch.float32, 768)])
def test_matches_64_bits(n, q, k, dtype, d):
    if n * d > 50_000_000:
        d = 64 if dtype == torch.float32 else 128
    docs, queries = _unit(n, d, 0).to(dtype), _unit(q, d, 1).to(dtype)
    values, indices = ops.knn_topk(queries, docs, k)
    exact = queries.double() @ docs.double().t()
    want = exact.topk(min(k, n), -1).values
    assert values.shape == indices.shape == want.shape
    # fp32 sums of d products of unit vectors' elements: below sqrt(d) 2^-24 by far
    assert (values.double() - want).abs().max() < 2 ** -20
    assert (exact.gather(1, indices) - want).abs().max() < 2 ** -20
    assert all(len(set(row)) == len(row) for row in indices.tolist())
    assert (values[:, 1:] <= values[:, :-1]).all()


@pytest.mark.parametrize("n", [40, 3000, 200000])
@pytest.mark.parametrize("k", [5, 64])
def test_equal_scores(n, k):
    """Equal documents: any k of the equal ones, each once."""
    docs = _unit(1, 64, 2).expand(n, 64).contiguous()
    docs[n // 2] *= 2
    values, indices = ops.knn_topk(docs[:1], docs, k)
    k = min(k, n)
    assert indices[0, 0] == n // 2
    assert len(set(indices[0].tolist())) == k and 0 <= indices.min() and indices.max() < n
    assert (values[0, 1:] - 1).abs().max() < 2 ** -20


def test_special_values():
    docs = _unit(3000, 64, 3)
    docs[7], docs[1999], docs[2500] = float("nan"), float("inf"), float("-inf")
    query = torch.ones(1, 64, device="cuda")
    values, indices = ops.knn_topk(query, docs, 64)
    want = (query @ docs.t()).topk(64, -1)
    assert torch.isnan(values[0, 0]) and torch.equal(indices[0, :2], want.indices[0, :2])
    assert values[0, 1] == float("inf") and torch.isfinite(values[0, 2:]).all()


@torch.inference_mode()  # as the engine captures: the generator is shared
def test_replay():
    docs, queries = _unit(40000, 128, 4), _unit(2, 128, 5)
    ops.knn_topk(queries, docs, 20)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.knn_topk(queries, docs, 20)
    for seed in (6, 7, 8):
        queries.copy_(_unit(2, 128, seed))
        graph.replay()
        want = ops.knn_topk(queries, docs, 20)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
