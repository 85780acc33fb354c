"""Prompt attention of few rows behind long contexts, whose keys are cut into parts."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu
P = 64


def _case(lens, past, hq, hkv, D, dtype, width=0):
    g = torch.Generator().manual_seed(sum(lens) + sum(past) + D)
    ctx = [a + b for a, b in zip(lens, past)]
    pages = [-(-c // P) for c in ctx]
    caches = [torch.randn(sum(pages) + 1, hkv, P, D, generator=g).to(dtype) for _ in range(2)]
    order = torch.randperm(sum(pages), generator=g) + 1
    bt, a = torch.zeros(len(lens), max(max(pages), width), dtype=torch.int32), 0
    for i, n in enumerate(pages):
        bt[i, :n] = order[a:a + n].int()
        a += n
    q = torch.randn(sum(lens), hq, D, generator=g).bfloat16()
    cu = torch.tensor([0, *lens]).cumsum(0).int()
    return [t.cuda() for t in (q, *caches, bt, cu, torch.tensor(ctx, dtype=torch.int32))]


def _want(q, kc, vc, bt, cu, ctx, scale):
    """In 64 bits, and what 16-bit weights and a rounded result may be off by."""
    outs, offs = [], []
    G = q.shape[1] // kc.shape[1]
    for s in range(len(ctx)):
        L, n = int(ctx[s]), int(cu[s + 1] - cu[s])
        rows = bt[s, :-(-L // P)].long()
        k, v = (c[rows].double().transpose(0, 1).reshape(c.shape[1], -1, c.shape[3])[:, :L]
                .repeat_interleave(G, 0) for c in (kc, vc))
        x = q[int(cu[s]):int(cu[s + 1])].double().transpose(0, 1) @ k.transpose(1, 2) * scale
        seen = torch.arange(L, device="cuda") <= torch.arange(L - n, L, device="cuda")[:, None]
        p = x.masked_fill(~seen, -torch.inf).softmax(-1)
        outs.append((p @ v).transpose(0, 1))
        offs.append((p @ v.abs()).transpose(0, 1))
    return torch.cat(outs), torch.cat(offs)


@pytest.mark.parametrize("lens,past", [
    ([1], [1500]), ([20], [700]), ([33], [12 * 64 - 33]), ([64], [13 * 64 - 64]),
    ([65], [5000]), ([300], [1029]), ([500], [1300]), ([1000], [2100]),
    ([60, 1, 70, 129], [4000, 30, 0, 900]), ([200, 100, 30], [0, 2000, 1])])
@pytest.mark.parametrize("hq,hkv,D", [(32, 8, 128), (32, 8, 64), (28, 4, 128), (6, 6, 64),
                                      (8, 4, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_against_64_bits(lens, past, hq, hkv, D, dtype):
    """Around the least number of tiles (12 and an eighth of the blocks), parts of six tiles and
    more, contexts that stay whole beside others that do not."""
    for width in (0, 200):
        q, kc, vc, bt, cu, ctx = _case(lens, past, hq, hkv, D, dtype, width)
        into = torch.empty_like(q)
        got = ops.attention_prefill_paged(q, kc, vc, bt, cu, ctx, D ** -0.5)
        ops.attention_prefill_paged(q, kc, vc, bt, cu, ctx, D ** -0.5, out=into)
        assert torch.equal(got, into)
        want, off = _want(q, kc, vc, bt, cu, ctx, D ** -0.5)
        # bf16 has 8 bits: a weight is rounded by up to 2^-8 of itself, the result of weights so
        # rounded once more by as much; fp32 sums are far below
        near = 2 ** -8 * off
        assert ((got.double() - want).abs() <= near + 2 ** -8 * (want.abs() + near) + 1e-6).all()


def test_cut_or_whole():
    """A row's result does not hang on how its keys are cut by more than roundings: alone, and
    among so many rows that contexts stay whole."""
    q, kc, vc, bt, cu, ctx = _case([64], [6000], 32, 8, 128, torch.bfloat16)
    one = ops.attention_prefill_paged(q, kc, vc, bt, cu, ctx, 128 ** -0.5)
    many = ops.attention_prefill_paged(
        q.repeat(40, 1, 1), kc, vc, bt.repeat(40, 1),
        torch.arange(41, dtype=torch.int32, device="cuda") * 64, ctx.repeat(40), 128 ** -0.5)
    assert torch.equal(many[:64], many[-64:])
    assert (one.float() - many[:64].float()).norm() <= 2 ** -7 * one.float().norm()


def test_eight_bits_stay_whole():
    """What an 8-bit cache's next rows are made of does not hang on other sequences."""
    q, kc, vc, bt, cu, ctx = _case([64], [6000], 32, 8, 128, torch.float8_e4m3fn)
    one = ops.attention_prefill_paged(q, kc, vc, bt, cu, ctx, 128 ** -0.5)
    many = ops.attention_prefill_paged(
        q.repeat(40, 1, 1), kc, vc, bt.repeat(40, 1),
        torch.arange(41, dtype=torch.int32, device="cuda") * 64, ctx.repeat(40), 128 ** -0.5)
    assert torch.equal(one, many[:64]) and torch.equal(one, many[-64:])


@pytest.mark.parametrize("mode,eight,steady", [("prefill", True, True), ("mixed", True, True),
                                               ("prefill", False, False), ("decode", True, False)])
def test_prompts_into_eight_bits(mode, eight, steady, monkeypatch):
    """A step's products keep their order of sums where its prompts fill an 8-bit cache."""
    from aurora_amd.models.config import ModelSpec
    from aurora_amd.models.llama import AttnMetadata, LlamaForCausalLM
    spec = ModelSpec(name="t", vocab_size=64, hidden_size=256, n_layers=2, n_heads=4,
                     n_kv_heads=2, head_dim=64, intermediate_size=512)
    model = LlamaForCausalLM(spec, device="cuda")
    model.init_random(0)
    dtype = torch.float8_e4m3fn if eight else torch.bfloat16
    caches = [tuple(torch.zeros(3, 2, P, 64, device="cuda").to(dtype) for _ in "kv")] * 2
    ints = [torch.tensor(v, dtype=torch.int32, device="cuda")
            for v in ([0, 1, 2], [P, P + 1, P + 2], [[1, 0]], [3], [0, 3])]
    if mode == "decode":
        ints[2], ints[3] = ints[2].repeat(3, 1), ints[3].repeat(3)
    meta = AttnMetadata(mode, *ints[:4], ints[4], num_prefill_tokens=3,
                        dec_block_tables=ints[2][:0], dec_context_lens=ints[3][:0])
    seen, real = [], ops.linear_parts
    monkeypatch.setattr(ops, "linear_parts",
                        lambda x, w, s=False: seen.append(s) or real(x, w, s))
    model(torch.tensor([1, 2, 3], device="cuda"), caches, meta)
    assert seen == [steady] * 6
