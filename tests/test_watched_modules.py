"""Modules that a user watches or replaces are called, and see whole results."""
import collections
import dataclasses
import types

import pytest
import torch
import torch.nn as nn

from aurora_amd.models.config import get_spec
from aurora_amd.models.encoder import SentenceEncoder
from aurora_amd.models.llama import AttnMetadata, LlamaForCausalLM

SPECS = {m: get_spec(m) for m in ("tiny-llama", "tiny-moe")}
DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


def _model(name, device, cls=LlamaForCausalLM):
    dtype = torch.bfloat16 if device == "cuda" else torch.float32
    spec = get_spec("smoke-moe" if name == "tiny-moe" else "smoke-llama") if device == "cuda" \
        else SPECS[name]
    m = cls(spec, dtype, device)
    m.init_random(1)
    return m


def _step(m, T):
    """The hidden states of one prompt of T tokens."""
    spec, dev, P = m.spec, m.embed.weight.device, 64
    caches = [tuple(torch.zeros(2, spec.n_kv_heads, P, spec.head_dim, dtype=m.dtype, device=dev)
                    for _ in range(2)) for _ in range(spec.n_layers)]
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    at = torch.arange(T, dtype=torch.int32, device=dev)
    meta = AttnMetadata(mode="prefill", positions=at, slot_mapping=at,
                        block_tables=i32(0, 1)[None], context_lens=i32(T),
                        cu_seqlens_q=i32(0, T))
    return m(torch.arange(T, device=dev) % 50, caches, meta)


def _decode(m, kind, n=3, past=40):
    """The hidden states of one token each behind n contexts."""
    spec, dev, P = m.spec, m.embed.weight.device, 64
    g = torch.Generator().manual_seed(n)
    caches = [tuple(torch.randn(2 * n * 8, spec.n_kv_heads, P, spec.head_dim, generator=g)
                    .to(dev, m.dtype) for _ in range(2)) for _ in range(spec.n_layers)]
    at = torch.full((n,), past, dtype=torch.int32, device=dev)
    tables = torch.arange(16 * n, dtype=torch.int32, device=dev).view(n, 16)
    return m(torch.arange(n, device=dev), caches, kind(
        mode="decode", positions=at, slot_mapping=tables[:, past // P] * P + past % P,
        block_tables=tables, context_lens=at + 1))


@dataclasses.dataclass
class _Counted(AttnMetadata):
    layers: int = dataclasses.field(default=0, init=False)


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("kind", [types.SimpleNamespace, _Counted, collections.namedtuple(
    "Step", "mode positions slot_mapping block_tables context_lens")])
def test_metadata_of_another_kind(device, kind):
    """What has the fields that a decoding step reads will do; contexts are cut or may be."""
    m = _model("tiny-llama", device)
    _same(_decode(m, kind, past=900), _decode(m, AttnMetadata, past=900))


def _same(a, b):
    """Equal on the CPU; on the GPU a watched module's own call may add up its bf16 products
    in another order, some 2^-9 of the stream for each of at most 12 layers' products."""
    if a.is_cuda:
        assert (a.double() - b.double()).norm() <= 2 ** -6 * b.double().norm()
    else:
        assert torch.equal(a, b)


WATCHED = ["layers.0", "layers.1", "layers.0.attn", "layers.0.attn.qkv_proj",
           "layers.1.attn.o_proj", "layers.0.mlp", "layers.0.mlp.gate_up", "layers.1.mlp.down"]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("name", WATCHED)
@pytest.mark.parametrize("T", [21, 1])  # of one row norms may be left to products
def test_hooks_of_decoders(name, device, T):
    m = _model("tiny-llama", device)
    before = _step(_model("tiny-llama", device), T)
    seen = []

    def look(module, args, out):
        for x in (*args[:1], out[0] if isinstance(out, tuple) else out):
            assert x.dim() == 2 and x.shape[0] == T and x.dtype == m.dtype
        seen.append(out)

    m.get_submodule(name).register_forward_hook(look)
    _same(_step(m, T), before)
    assert len(seen) == 1


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("name", ["attn.qkv_proj", "attn.o_proj", "mlp.gate_up", "mlp.down"])
@pytest.mark.parametrize("T", [21, 1])
def test_replaced_projections(name, device, T):
    """An adapter in place of a projection, a forward of the instance's own."""
    m, way = _model("tiny-llama", device), _model("tiny-llama", device)

    class Doubled(nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, x):
            return 2 * self.inner(x)

    parent, _, child = f"layers.1.{name}".rpartition(".")
    setattr(m.get_submodule(parent), child, Doubled(m.get_submodule(f"{parent}.{child}")))
    own = way.get_submodule(f"{parent}.{child}")
    own.forward = lambda x, f=own.forward: 2 * f(x)
    plain = _model("tiny-llama", device)
    plain.get_submodule(f"{parent}.{child}").weight.data.mul_(2)  # exact
    want = _step(plain, T)
    plain = _step(_model("tiny-llama", device), T)
    assert (plain - want).norm() > 2 ** -4 * want.norm()
    _same(_step(m, T), want)
    _same(_step(way, T), want)


@pytest.mark.parametrize("device", DEVICES)
def test_hooks_of_routed_models(device):
    m = _model("tiny-moe", device)
    seen = []
    for name in ("layers.0.mlp", "layers.0.mlp.router", "layers.1.mlp.router"):
        m.get_submodule(name).register_forward_hook(lambda *a, n=name: seen.append(n))
    for e in m.layers[1].mlp.experts:
        e.register_forward_hook(lambda *a: seen.append("expert"))
    _step(m, 100)
    assert seen[:3] == ["layers.0.mlp.router", "layers.0.mlp", "layers.1.mlp.router"]
    seen.clear()
    m.layers[1].mlp(torch.randn(300, m.spec.hidden_size, device=device).to(m.dtype))
    assert seen.count("expert") >= 2


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("name", ["layers.0", "layers.1", "layers.0.gate_up", "layers.1.down",
                                  "layers.1.qkv"])
def test_hooks_of_encoders(name, device):
    spec = "tiny-encoder" if device == "cpu" else "bge-base"
    torch.manual_seed(0)
    m = SentenceEncoder(spec, device=device)
    m.init_random(2)
    texts = [[5, 6, 7], list(range(40))]
    before = m.encode_ids(texts)
    seen = []
    m.get_submodule(name).register_forward_hook(lambda mod, args, out: seen.append(out))
    _same(m.encode_ids(texts), before)
    assert len(seen) == 1 and seen[0].dim() == 2 and seen[0].shape[0] == 43
    layer, x = m.layers[0], torch.randn(43, m.spec.hidden_size, device=device)
    out = layer(x.to(m.embed.weight.dtype), m.cos_sin,  # called as a layer by itself
                torch.arange(43, dtype=torch.int32, device=device),
                torch.tensor([0, 43], dtype=torch.int32, device=device))
    assert out.shape == x.shape


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("texts", [[[5]], [[5, 6, 7], [8], list(range(1, 30))]])
def test_encoders_leave_what_is_not_theirs(device, texts):
    """What a hook keeps of the joint projection stays as it was, and a tensor that somebody
    hands back on every pass gives the same embeddings on every pass."""
    m = SentenceEncoder("tiny-encoder" if device == "cpu" else "bge-base", device=device)
    m.init_random(1)
    before, kept = m.encode_ids(texts), []
    hook = m.layers[0].qkv.register_forward_hook(
        lambda module, args, out: kept.append((out, out.clone())))
    _same(m.encode_ids(texts), before)
    assert torch.equal(*kept[0])
    hook.remove()
    m.layers[0].qkv.forward = lambda x, made=kept[0][1]: made
    for _ in range(3):
        _same(m.encode_ids(texts), before)
