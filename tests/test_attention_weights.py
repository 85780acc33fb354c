"""Softmax weights of the attention kernels that multiply in fp32: how many bits they keep,
and what infinite and unseen values do to them."""
import pytest
import torch

from aurora_amd import ops
from aurora_amd.ops.sequence import Segment, biased_attention

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def _near(D):
    """Of every sequence three keys: one with most of the weight and value 0, two whose
    weights differ by 2^-13 of themselves and whose values are 1 and -1."""
    s = ((torch.arange(128) + 128) / 128 * 2 ** -6).bfloat16()
    k = torch.zeros(128, 3, D).bfloat16()
    k[:, :, 0] = torch.stack([s + 1, s, s + 2 ** -13], 1)
    v = torch.tensor([0.0, 1.0, -1.0]).view(1, 3, 1).expand(128, 3, D).bfloat16()
    w = k[:, :, 0].double().softmax(1)
    return k, v, (w[:, 1] - w[:, 2]).view(128, 1, 1)


def _check_near(out, want):
    # bf16's rounding, and of terms of at most 0.27 an fp32 exponential's, scores' and sums'
    # errors, some units of 2^-25 each; weights of 17 bits are off by up to 2^-19
    assert ((out.double().cpu() - want).abs() <= want.abs() * 2 ** -8 + 2 ** -22).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("P", [16, 64])
def test_decoding_keeps_32_bits(D, P):
    k, v, want = _near(D)
    kc, vc = (torch.zeros(128, 1, P, D).bfloat16() for _ in range(2))
    kc[:, 0, :3], vc[:, 0, :3] = k, v
    q = torch.zeros(128, 2, D).bfloat16()
    q[:, :, 0] = 1
    bt = torch.arange(128, dtype=torch.int32)[:, None]
    out = ops.paged_attention_decode(q.cuda(), kc.cuda(), vc.cuda(), bt.cuda(),
                                     torch.full((128,), 3, dtype=torch.int32).cuda(), 1.0)
    _check_near(out, want)


def _decode(L, P, D, B=3, bias=False, window=0, spoil=None, cache=torch.bfloat16):
    """Decoding over L cached tokens, some rows of the cache spoiled -> outputs, weights,
    values."""
    g = torch.Generator().manual_seed(L)
    n = -(-L // P)
    kc, vc = (torch.randn(B * n, 2, P, D, generator=g) for _ in range(2))
    q = torch.randn(B, 4, D, generator=g).bfloat16()
    bt = torch.arange(B * n, dtype=torch.int32).view(B, n)
    spoil(kc.view(B, n, 2, P, D), vc.view(B, n, 2, P, D))
    kc, vc = kc.to(cache), vc.to(cache)
    args = [x.cuda() for x in (kc, vc, bt, torch.full((B,), L, dtype=torch.int32))]
    if bias:
        seg = Segment(rows=slice(0, B), block_tables=args[2], context_lens=args[3],
                      starts=args[3] - 1, state_slots=None)
        out = torch.empty(B, 4 * D, dtype=torch.bfloat16, device="cuda")
        biased_attention(q.cuda(), args[0], args[1], seg, D ** -0.5, window, None, out, 0, D, 1.0)
        out = out.view(B, 4, D)
    else:
        out = ops.paged_attention_decode(q.cuda(), *args, D ** -0.5)
    first = max(0, L - window) if window else 0
    keys, values = (x.float().view(B, n, 2, P, D).transpose(2, 3).reshape(B, n * P, 2, D)
                    [:, first:L].repeat_interleave(2, 2).double() for x in (kc, vc))
    w = torch.softmax((keys * q[:, None].double()).sum(-1) * D ** -0.5, 1)
    want = (w[..., None] * values).sum(1)
    return out.double().cpu(), want


def _check(out, want):
    assert torch.equal(out.isnan(), want.isnan())
    assert torch.equal(out.isposinf(), want.isposinf())
    assert torch.equal(out.isneginf(), want.isneginf())
    ok = want.isfinite()
    assert (out - want)[ok].norm() <= 2 ** -8 * want[ok].norm()


@pytest.mark.parametrize("L,P", [(1, 16), (40, 16), (40, 64), (300, 64), (2000, 256)])
@pytest.mark.parametrize("D", [64, 128])
def test_decoding_over_infinite_values(L, P, D):
    def spoil(kc, vc):
        vc[0, 0, 0, 0, 3] = INF           # seen: the channel is infinite, its neighbours not
        vc[1, (L - 1) // P, 1, (L - 1) % P, 5] = -INF
        vc[2, 0, 0, 0, 7] = NAN
    _check(*_decode(L, P, D, spoil=spoil))


@pytest.mark.parametrize("L,P", [(1, 16), (40, 16), (40, 64), (300, 64), (2000, 256)])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn])
def test_decoding_beside_spoiled_rows(L, P, cache):
    def spoil(kc, vc):
        for c in (kc, vc):
            c[:, -1, :, (L - 1) % P + 1:] = NAN  # rows past the context
    _check(*_decode(L, P, 64, spoil=spoil, cache=cache))


@pytest.mark.parametrize("L,window", [(200, 70), (300, 1), (1999, 1024)])
def test_decoding_behind_a_window(L, window):
    def spoil(kc, vc):
        for c in (kc, vc):
            first = L - window
            c[:, first // 64, :, :first % 64] = INF  # rows before the window
            c[:, -1, :, (L - 1) % 64 + 1:] = -INF
    _check(*_decode(L, 64, 64, bias=True, window=window, spoil=spoil))


@pytest.mark.parametrize("P", [16, 48, 64])
@pytest.mark.parametrize("L,window", [(100, 1), (200, 70), (203, 120)])
def test_decoding_without_the_pages_behind_a_window(P, L, window):
    """The block table need not name pages that nobody sees."""
    g = torch.Generator().manual_seed(L)
    n = -(-L // P)
    kc, vc = (torch.randn(n, 2, P, 64, generator=g).bfloat16().cuda() for _ in range(2))
    q = torch.randn(1, 4, 64, generator=g).bfloat16().cuda()
    ctx = torch.tensor([L], dtype=torch.int32, device="cuda")
    results = []
    for hidden in (0, -1):
        bt = torch.arange(n, dtype=torch.int32, device="cuda")[None].clone()
        bt[:, :(L - window) // P] = hidden
        seg = Segment(rows=slice(0, 1), block_tables=bt, context_lens=ctx, starts=ctx - 1,
                      state_slots=None)
        results.append(torch.empty(1, 256, dtype=torch.bfloat16, device="cuda"))
        biased_attention(q, kc, vc, seg, 0.125, window, None, results[-1], 0, 64, 1.0)
    assert torch.equal(*results) and results[0].isfinite().all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_packed_rows_keep_32_bits(D, causal):
    k, v, want = _near(D)
    q = torch.zeros(128 * 3, 1, D).bfloat16()
    q[:, :, 0] = 1
    cu = torch.arange(129, dtype=torch.int32) * 3
    out = ops.attention_prefill(q.cuda(), k.reshape(-1, 1, D).cuda(), v.reshape(-1, 1, D).cuda(),
                                cu.cuda(), 1.0, causal=causal)
    _check_near(out.view(128, 3, D)[:, 2:], want)  # the last row sees all three


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("value", [INF, -INF, NAN])
def test_packed_rows_over_infinite_values(D, causal, value):
    """Only rows that see an infinite value are infinite in its channel, in every place of
    a tile, at a sequence's end and beside other sequences."""
    g = torch.Generator().manual_seed(D)
    lens = [1, 31, 40, 64, 65, 100, 130, 200]
    at = [0, 30, 39, 17, 64, 70, 33, 131]  # the spoiled row of each
    cu = torch.tensor([0] + lens).cumsum(0)
    T = int(cu[-1])
    q, k, v = (torch.randn(T, h, D, generator=g).bfloat16() for h in (4, 2, 2))
    for s, a in enumerate(at):
        v[cu[s] + a, s % 2, (7 * s) % D] = value
    out = ops.attention_prefill(*(x.cuda() for x in (q, k, v)), cu.int().cuda(), D ** -0.5,
                                causal=causal).double().cpu()
    want = torch.empty(T, 4, D, dtype=torch.float64)
    for s, n in enumerate(lens):
        rows = slice(int(cu[s]), int(cu[s + 1]))
        x, keys, values = (t[rows].double().transpose(0, 1) for t in (
            q, k.repeat_interleave(2, 1), v.repeat_interleave(2, 1)))
        w = x @ keys.transpose(1, 2) * D ** -0.5
        for r in range(n):
            sees = r + 1 if causal else n
            p = w[:, r, :sees].softmax(-1)
            want[rows.start + r] = (p[:, :, None] * values[:, :sees]).sum(1)
    _check(out, want)
