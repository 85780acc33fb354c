"""Calls that autograd, a transform or a trace follows still give what they gave."""
import pytest
import torch
import torch.autograd.forward_ad as fwd

from aurora_amd import ops

pytestmark = pytest.mark.gpu


def _search_inputs():
    g = torch.Generator().manual_seed(3)
    return (torch.randn(*s, generator=g).cuda() for s in ((4, 256), (500, 256)))


def test_search_gradients():
    q, d = _search_inputs()
    q.requires_grad_(), d.requires_grad_()
    values, index = ops.knn_topk(q, d, 5)
    values.sum().backward()
    with torch.no_grad():
        want = torch.zeros_like(d).index_add_(0, index.flatten(), q.repeat_interleave(5, 0))
        torch.testing.assert_close(q.grad, d[index].sum(1), rtol=1e-5, atol=1e-4)
        torch.testing.assert_close(d.grad, want, rtol=1e-5, atol=1e-4)
        plain, where = ops.knn_topk(q, d, 5)  # nobody follows: the kernel
    torch.testing.assert_close(values.detach(), plain, rtol=1e-5, atol=1e-4)
    assert torch.equal(index, where)


def test_search_transforms():
    q, d = _search_inputs()
    values, index = ops.knn_topk(q, d, 5)
    mapped = torch.func.vmap(lambda x: ops.knn_topk(x[None], d, 5)[0][0])(q)
    torch.testing.assert_close(mapped, values, rtol=1e-5, atol=1e-4)
    grad = torch.func.grad(lambda x: ops.knn_topk(x, d, 5)[0].sum())(q)
    torch.testing.assert_close(grad, d[index].sum(1), rtol=1e-5, atol=1e-4)
    with fwd.dual_level():
        out = ops.knn_topk(fwd.make_dual(q, torch.ones_like(q)), d, 5)[0]
        tangent = fwd.unpack_dual(out).tangent
    torch.testing.assert_close(tangent, d[index].sum(-1), rtol=1e-5, atol=1e-3)


def test_search_traced():
    q, d = _search_inputs()
    traced = torch.jit.trace(lambda x: ops.knn_topk(x, d, 5)[0], q, check_trace=False)
    torch.testing.assert_close(traced(-q), ops.knn_topk(-q, d, 5)[0], rtol=1e-5, atol=1e-4)
