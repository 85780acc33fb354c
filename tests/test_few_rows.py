"""Products of few rows at the edges of their tiles, stages and parts, and their readers."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu

M = [1, 16, 32, 33, 64, 65, 96, 97, 128]
#: columns: tiles of 64 (32 of silu's outputs), four outputs a lane; K: one stage to
#: more than a ring of them
SHAPES = [(8, 64), (63, 128), (65, 192), (200, 448), (96, 1024), (1000, 576), (4096, 512)]


def _inputs(m, n, k, seed=0):
    g = torch.Generator().manual_seed(seed)
    x, w = (torch.randn(r, k, generator=g).bfloat16().cuda() for r in (m, n))
    return x, w * k ** -0.5


def _check(got, want, k):
    """The result in 64 bits rounded to bf16, but for K fp32 sums of terms of size about
    |want| / sqrt(K): far below 2^-16 of the largest, which moves some to the other
    neighbour."""
    assert torch.isfinite(got).all()
    slack = 2 ** -16 * want.abs().max()
    assert ((got.double() - want).abs() <= want.abs() * 2 ** -8 + slack).all()


@pytest.mark.parametrize("m", M)
@pytest.mark.parametrize("n,k", SHAPES)
def test_products(m, n, k):
    from aurora_amd import _hip_ops
    x, w = _inputs(m, n, k)
    want = x.double() @ w.double().t()
    for parts in (1, 2, 3, 7, 16):
        _check(_hip_ops.few_rows(x, w, False, parts), want, k)
        raw = _hip_ops.few_rows(x, w, True, parts)
        _check((raw.sum(0) if raw.dim() == 3 else raw).bfloat16(), want, k)
    _check(ops.linear(x, w), want, k)


@pytest.mark.parametrize("m", M)
@pytest.mark.parametrize("n,k", [(4, 64), (31, 128), (33, 192), (100, 448), (48, 1024),
                                 (12352, 384)])
def test_silu(m, n, k):
    x, w = _inputs(m, 2 * n, k)
    y = x.double() @ w.double().t()
    want = torch.nn.functional.silu(y[:, :n]) * y[:, n:]
    from aurora_amd import _hip_ops
    _check(_hip_ops.silu_few_rows(x, w), want, k)
    if n % 8 == 0:  # as silu_mul by itself
        _check(ops.linear_silu_mul(x, w), want, k)


@pytest.mark.parametrize("m", [1, 33, 128])
@pytest.mark.parametrize("n", [64, 1024, 4096, 10240])
@pytest.mark.parametrize("parts", [2, 7, 16])
def test_norm_of_parts(m, n, parts):
    g = torch.Generator().manual_seed(1)
    raw = torch.randn(parts, m, n, generator=g).cuda()
    res, weight = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((m, n), (n,)))
    total = raw[0].clone()
    for p in raw[1:]:
        total += p
    got, got_res = ops.rmsnorm_residual(raw, res, weight, 1e-5)
    want, want_res = ops.rmsnorm_residual(total.bfloat16(), res, weight, 1e-5)
    assert torch.equal(got_res, want_res)
    # the row's fp32 sum of squares is added up in another order
    assert ((got.float() - want.float()).abs() <= want.float().abs() * 2 ** -7).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("parts", [1, 3, 16])
@pytest.mark.parametrize("biased", [False, True])
def test_rotation_of_parts(D, dtype, parts, biased):
    g = torch.Generator().manual_seed(2)
    T, hq, hkv, P = 9, 6, 2, 16
    width = (hq + 2 * hkv) * D
    raw = torch.randn(parts, T, width, generator=g).cuda()
    bias = torch.randn(width, generator=g).bfloat16().cuda()
    total = raw[0].clone()
    for p in raw[1:]:
        total += p
    plain = total.bfloat16()
    cs = ops.torch_ref.rope_cos_sin_cache(D, 64, 10000.0, dtype=torch.float32).cuda()
    at = torch.arange(T, dtype=torch.int32, device="cuda")
    slots = at * 3 % 32
    slots[4] = -1
    results = []
    for qkv, b in ((raw, bias if biased else None), (plain + bias if biased else plain, None)):
        caches = [torch.zeros(2, hkv, P, D, device="cuda").to(dtype) for _ in range(2)]
        q = ops.fused_rope_kv_write(qkv, at, slots, cs, *caches, hq, hkv, b)
        results.append([q] + [c.float() for c in caches])
    for a, b in zip(*results):
        assert torch.equal(a, b)
    if biased:  # a plain product with its bias in the same kernel
        caches = [torch.zeros(2, hkv, P, D, device="cuda").to(dtype) for _ in range(2)]
        q = ops.fused_rope_kv_write(plain, at, slots, cs, *caches, hq, hkv, bias)
        for a, b in zip([q] + [c.float() for c in caches], results[0]):
            assert torch.equal(a, b)


@pytest.mark.parametrize("D,T", [(128, 230), (64, 460), (72, 3), (24, 5), (128, 2000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_rotation_widths(D, T, dtype):
    """Eight columns a thread from 2^20 values on, one below and for other widths."""
    g = torch.Generator().manual_seed(D)
    hq, hkv, P = 32, 2, 16
    qkv = torch.randn(T, (hq + 2 * hkv) * D, generator=g).bfloat16()
    cs = ops.torch_ref.rope_cos_sin_cache(D, T, 10000.0, dtype=torch.float32)
    at = torch.arange(T, dtype=torch.int32)
    slots = torch.randperm(-(-T // P) * P, generator=g)[:T].int()
    slots[T // 2] = -1
    kc, vc = (torch.zeros(-(-T // P), hkv, P, D).to(dtype).cuda() for _ in range(2))
    q = ops.fused_rope_kv_write(qkv.cuda(), at.cuda(), slots.cuda(), cs.cuda(), kc, vc, hq, hkv)
    k_want, v_want = torch.zeros(kc.shape), torch.zeros(kc.shape)
    keep = slots >= 0
    q_want = ops.fused_rope_kv_write(qkv[keep].float(), at[keep], slots[keep], cs, k_want,
                                     v_want, hq, hkv)
    # rounded once, to 2^-8 or to 2^-4 of itself (or half the 8-bit type's smallest step)
    for got, want, step in ((q.cpu()[keep], q_want, 2 ** -8),
                            (kc.cpu(), k_want, 2 ** -8 if dtype == torch.bfloat16 else 2 ** -4),
                            (vc.cpu(), v_want, 2 ** -8 if dtype == torch.bfloat16 else 2 ** -4)):
        assert ((got.float() - want).abs() <= step * want.abs() + 2 ** -10).all()


@pytest.mark.parametrize("M", [1, 2, 33, 65, 128])
@pytest.mark.parametrize("step,first", [(256, 64), (200, 8), (136, 0), (131, 0), (256, 3)])
def test_strided_rows(M, step, first):
    """Columns of a wider tensor, at distances and addresses that 16-byte loads can read and
    at others."""
    from aurora_amd import _hip_ops
    K, N = 128, 96
    x = torch.randn(M, step + 64, device="cuda").bfloat16().as_strided((M, K), (step, 1), first)
    w = torch.randn(2 * N, K, device="cuda").bfloat16()
    whole = x.contiguous().clone()
    for parts in (1, 2):
        assert torch.equal(_hip_ops.few_rows(x, w, False, parts),
                           _hip_ops.few_rows(whole, w, False, parts))
    assert torch.equal(_hip_ops.silu_few_rows(x, w), _hip_ops.silu_few_rows(whole, w))
    assert torch.equal(ops.linear(x, w), ops.linear(whole, w))
