"""Stretches of a context, merged by the workgroup that ends last."""
import pytest
import torch

from aurora_amd import ops
from test_decode_stretches import _case, _check, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stretches", [1, 2, 8, 9, 31, 32, 33, 40])
@pytest.mark.parametrize("H,G,D", [(4, 4, 64), (1, 1, 128), (7, 7, 128), (17, 17, 64)])
def test_as_many(stretches, H, G, D):
    """Around what is read at once; heads that leave half a wave idle, more than a tile has."""
    args = _case([128 * stretches - 5], 256, H, G, D, torch.bfloat16, room=8192)
    marks = ops.decode_marks(H, args[1], args[3])
    assert marks is not None
    for _ in range(3):  # marks are left as they were found
        out = torch.full_like(args[0], float("nan"))
        ops.paged_attention_decode(*args, D ** -0.5, out=out, marks=marks)
        _check(out, _reference(*args, D ** -0.5))
        assert not marks.any()


@pytest.mark.parametrize("marks", ["none", "too few", "of another type"])
def test_without_marks(marks):
    """A call that brings none that fit makes its own; the sequences' numbers of stretches
    differ, and one sequence stands twice in the batch."""
    q, k, v, bt, ctx = _case([1, 5000, 129, 700, 2500], 64, 8, 4, 128, torch.bfloat16)
    q, bt, ctx = q[[0, 1, 2, 1, 3, 4]], bt[[0, 1, 2, 1, 3, 4]], ctx[[0, 1, 2, 1, 3, 4]]
    fit = {"none": None, "too few": torch.zeros(3, dtype=torch.int32, device="cuda"),
           "of another type": torch.zeros(99, device="cuda")}[marks]
    _check(ops.paged_attention_decode(q, k, v, bt, ctx, 0.08, marks=fit),
           _reference(q, k, v, bt, ctx, 0.08))


def test_captured():
    """A graph's marks are its own: every replay gives the eager result."""
    args = _case([900, 3000, 40], 64, 8, 4, 64, torch.bfloat16)
    want = ops.paged_attention_decode(*args, 0.125)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        marks = ops.decode_marks(8, args[1], args[3])
        for _ in range(2):
            out = ops.paged_attention_decode(*args, 0.125, marks=marks)
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(ops.paged_attention_decode(*args, 0.125), want)
