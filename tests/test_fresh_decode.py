"""Rotation, cache write and decode attention in one kernel."""
import pytest
import torch

from aurora_amd import ops

P = 32


def _case(B, contexts, hq, hkv, D, parts, biased, dtype, dev, MP=None):
    g = torch.Generator().manual_seed(B + hq + D + parts)
    width = (hq + 2 * hkv) * D
    ctx = torch.tensor([contexts[i % len(contexts)] for i in range(B)], dtype=torch.int32)
    pages = [-(-int(c) // P) for c in ctx]
    MP = MP or max(pages) + 1
    order = torch.randperm(sum(pages), generator=g) + 1
    bt = torch.zeros(B, MP, dtype=torch.int32)
    slots, a = [], 0
    for b, (c, n) in enumerate(zip(ctx.tolist(), pages)):
        bt[b, :n] = order[a:a + n].int()
        slots.append(int(bt[b, (c - 1) // P]) * P + (c - 1) % P)
        a += n
    caches = [torch.randn(sum(pages) + 1, hkv, P, D, generator=g).to(dtype) for _ in range(2)]
    for c in caches:  # what stood in the new rows' place does not matter
        raw = c.view(torch.uint8) if dtype != torch.bfloat16 else c.view(torch.int16)
        for s in slots:
            raw[s // P, :, s % P] = 0x7f if dtype != torch.bfloat16 else 0x7fc0
    qkv = torch.randn(parts or 1, B, width, generator=g) * (parts or 1) ** -0.5
    if not parts:
        qkv = qkv[0].bfloat16()
    bias = torch.randn(width, generator=g).bfloat16() if biased else None
    cs = ops.torch_ref.rope_cos_sin_cache(D, int(ctx.max()) + 1, 10000.0, dtype=torch.float32)
    return [t if t is None else t.to(dev) for t in
            (qkv, bias, ctx - 1, torch.tensor(slots, dtype=torch.int32), cs, *caches, bt, ctx)]


@pytest.mark.gpu
@pytest.mark.parametrize("contexts", [
    [1], [2, 31, 32, 33, 64, 65], [127, 128, 129, 1, 160, 480], [5000], [3000, 1, 700, 513],
    [512, 1024, 1536]])
@pytest.mark.parametrize("hq,hkv,D", [(32, 8, 128), (32, 8, 64), (28, 4, 128), (4, 4, 64),
                                      (40, 2, 128)])
@pytest.mark.parametrize("parts,biased,dtype", [
    (0, False, torch.bfloat16), (2, True, torch.bfloat16), (4, False, torch.float8_e4m3fn),
    (5, True, torch.float8_e4m3fn), (11, False, torch.bfloat16)])
def test_as_two_kernels(contexts, hq, hkv, D, parts, biased, dtype):
    """The same bits, in the caches too, whole contexts and cut ones."""
    for B, MP in ((len(contexts), None), (len(contexts), 512), (70, None)):
        qkv, bias, at, slots, cs, kc, vc, bt, ctx = _case(
            B, contexts, hq, hkv, D, parts, biased, dtype, "cuda", MP)
        marks = ops.decode_marks(hq, kc, bt)
        k2, v2 = kc.clone(), vc.clone()
        out = ops._hip.fresh_attention_decode(qkv, bias, cs, kc, vc, bt, ctx, hq, D ** -0.5,
                                              marks)
        assert out is not None
        q = ops.fused_rope_kv_write(qkv, at, slots, cs, k2, v2, hq, hkv, bias)
        want = ops.paged_attention_decode(q, k2, v2, bt, ctx, D ** -0.5, marks=marks)
        bits = torch.uint8 if dtype != torch.bfloat16 else torch.int16
        assert torch.equal(kc.view(bits), k2.view(bits)) and torch.equal(vc.view(bits),
                                                                         v2.view(bits))
        assert torch.isfinite(out).all()
        assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("B", [129, 170, 171, 192, 256, 257, 300])
@pytest.mark.parametrize("hq,hkv,D", [(32, 8, 128), (32, 8, 64), (28, 4, 128)])
@pytest.mark.parametrize("parts,biased,dtype", [
    (0, False, torch.bfloat16), (3, True, torch.bfloat16), (2, False, torch.float8_e4m3fn),
    (0, True, torch.float8_e4m3fn)])
def test_many_rows_as_two_kernels(B, hq, hkv, D, parts, biased, dtype):
    """The batches that are captured and more: the separate kernel has another order of sums from
    a million elements on (171 rows of 6144)."""
    contexts = [1 + 53 * i % 971 for i in range(B)]
    qkv, bias, at, slots, cs, kc, vc, bt, ctx = _case(
        B, contexts, hq, hkv, D, parts, biased, dtype, "cuda")
    k2, v2 = kc.clone(), vc.clone()
    out = ops._hip.fresh_attention_decode(qkv, bias, cs, kc, vc, bt, ctx, hq, D ** -0.5, None)
    q = ops.fused_rope_kv_write(qkv, at, slots, cs, k2, v2, hq, hkv, bias)
    want = ops.paged_attention_decode(q, k2, v2, bt, ctx, D ** -0.5)
    bits = torch.uint8 if dtype != torch.bfloat16 else torch.int16
    assert torch.equal(kc.view(bits), k2.view(bits)) and torch.equal(vc.view(bits), v2.view(bits))
    assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("idle", [1, 5, 130])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_idle_rows(idle, dtype):
    """Rows of a captured batch that no sequence fills are all alike, on one page with a context
    of one: the others and their pages are as without them."""
    B, hq, hkv, D = 60, 8, 2, 128
    qkv, _, at, slots, cs, kc, vc, bt, ctx = _case(
        B, [1, 31, 33, 700, 129], hq, hkv, D, 0, False, dtype, "cuda")
    k2, v2 = kc.clone(), vc.clone()
    want = ops.fresh_attention_decode(qkv, None, at, slots, cs, k2, v2, bt, ctx, hq, 0.1)
    more = lambda t, v: torch.cat([t, t.new_full((idle, *t.shape[1:]), v)])  # noqa: E731
    scratch = 0  # of the pages that _case gives to nobody
    out = ops.fresh_attention_decode(more(qkv, 0.5), None, more(at, 0), more(slots, scratch * P),
                                     cs, kc, vc, more(bt, scratch), more(ctx, 1), hq, 0.1)
    bits = torch.uint8 if dtype != torch.bfloat16 else torch.int16
    assert torch.equal(out[:B], want) and torch.isfinite(out).all()
    assert torch.equal(kc.view(bits)[1:], k2.view(bits)[1:])
    assert torch.equal(vc.view(bits)[1:], v2.view(bits)[1:])


@pytest.mark.gpu
def test_refused_forms_run_as_two():
    """Widths, pages and layouts without a form."""
    args = dict(parts=0, biased=False, dtype=torch.bfloat16, dev="cuda")
    for D, page in ((96, 32), (64, 16)):
        qkv, bias, at, slots, cs, kc, vc, bt, ctx = _case(3, [5, 9, 14], 4, 2, D, **args)
        kc, vc = (c.reshape(-1, 2, page, D).contiguous() if page == 32 else
                  c[:, :, :page].contiguous() for c in (kc, vc))
        slots = bt[:, 0] * page + ctx - 1
        assert ops._hip.fresh_attention_decode(qkv, bias, cs, kc, vc, bt, ctx, 4, 0.1,
                                               None) is None
        if D == 64:
            out = ops.fresh_attention_decode(qkv, bias, at, slots, cs, kc, vc, bt, ctx, 4, 0.1)
            assert torch.isfinite(out).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D,page", [(64, 16), (128, 16)])
def test_refused_pages(D, page):
    """Pages without a form: the reference's results and cache."""
    qkv, bias, at, slots, cs, kc, vc, bt, ctx = _case(3, [5, 9, 14], 4, 2, D, 0, True,
                                                      torch.bfloat16, "cuda")
    kc, vc = (c[:, :, :page].nan_to_num().contiguous() for c in (kc, vc))
    slots = bt[:, 0] * page + ctx - 1
    args = [qkv, bias, at, slots, cs, kc, vc, bt, ctx]
    host = [t.cpu() for t in args]
    assert ops._hip.fresh_attention_decode(qkv, bias, cs, kc, vc, bt, ctx, 4, 0.1, None) is None
    out = ops.fresh_attention_decode(*args, 4, 0.1).float().cpu()
    want = ops.fresh_attention_decode(*host, 4, 0.1).float()
    # a row may round the other way in bf16; of results as well, whose weights add up to one
    for got, held in ((kc, host[5]), (vc, host[6])):
        got, held = got.float().cpu(), held.float()
        assert ((got - held).abs() <= 2 ** -7 * held.abs() + 1e-6).all()
    assert ((out - want).abs() <= 2 ** -6 * host[6].float().abs().max()).all()


def test_reference():
    """Without a GPU: the two operations."""
    qkv, bias, at, slots, cs, kc, vc, bt, ctx = _case(3, [1, 33, 70], 4, 2, 64, 0, True,
                                                      torch.bfloat16, "cpu")
    k2, v2 = kc.clone(), vc.clone()
    out = ops.fresh_attention_decode(qkv, bias, at, slots, cs, kc, vc, bt, ctx, 4, 0.125)
    q = ops.fused_rope_kv_write(qkv, at, slots, cs, k2, v2, 4, 2, bias)
    assert torch.equal(out, ops.paged_attention_decode(q, k2, v2, bt, ctx, 0.125))
    assert torch.equal(kc, k2) and torch.equal(vc, v2)
