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


#: rows, outputs, K: what the kernels of few rows, of many and of prompts take otherwise
PRODUCTS = [(40, 256, 192), (100, 256, 3072), (300, 64, 64), (6400, 4096, 14336)]


@pytest.mark.parametrize("m,n,k", PRODUCTS)
def test_product_gradients(m, n, k):
    x = torch.randn(m, k, device="cuda").bfloat16().requires_grad_()
    w = (torch.randn(n, k, device="cuda") * k ** -0.5).bfloat16()
    y = ops.linear(x, w)
    y.backward(torch.ones_like(y))
    want = w.double().sum(0).expand(m, k)
    # sums of n terms, rounded to bf16
    assert (x.grad.double() - want).norm() <= 2 ** -7 * want.norm()


@pytest.mark.parametrize("m,n,k", PRODUCTS[:3])
def test_product_transforms(m, n, k):
    x = torch.randn(3, m, k, device="cuda").bfloat16()
    w = (torch.randn(n, k, device="cuda") * k ** -0.5).bfloat16()
    want = x.double() @ w.double().t()
    for f in (ops.linear, ops.linear_parts):
        got = torch.func.vmap(f, in_dims=(0, None))(x, w)
        assert (got.double() - want).norm() <= 2 ** -8 * want.norm()
    traced = torch.jit.trace(lambda a: ops.linear(a, w), x[0], check_trace=False)
    got = traced(x[1])
    assert (got.double() - want[1]).norm() <= 2 ** -8 * want[1].norm()


def test_products_of_two_devices():
    with pytest.raises(RuntimeError):
        ops.linear(torch.ones(4, 64, device="cuda").bfloat16(), torch.ones(8, 64).bfloat16())
