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
