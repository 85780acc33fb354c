"""Products on their way into an 8-bit cache keep their order of sums, whoever watches them."""
import types

import pytest
import torch
import torch.nn as nn

from aurora_amd import ops
from aurora_amd.models.config import ModelSpec
from aurora_amd.models.llama import AttnMetadata, LlamaForCausalLM, LlamaMLP

P = 64
GPU = pytest.mark.gpu


def _model(width=256, experts=0, device="cuda"):
    spec = ModelSpec(name="t", vocab_size=64, hidden_size=width, n_layers=2,
                     n_heads=width // 128 or 1, n_kv_heads=max(width // 512, 1), head_dim=128,
                     intermediate_size=512, n_experts=experts)
    m = LlamaForCausalLM(spec, torch.bfloat16 if device == "cuda" else torch.float32, device)
    m.init_random(0)
    return m


def _parts(m, T, eight=True, kind=AttnMetadata):
    """What a step of one prompt of T tokens is called with."""
    s, dev, n = m.spec, m.embed.weight.device, -(-T // P)
    dtype = torch.float8_e4m3fn if eight else m.dtype
    caches = [tuple(torch.zeros(n, s.n_kv_heads, P, s.head_dim, device=dev).to(dtype)
                    for _ in "kv") for _ in range(s.n_layers)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    at = i32(list(range(T)))
    return torch.arange(T, device=dev) % 64, caches, kind(
        mode="prefill", positions=at, slot_mapping=at, block_tables=i32([list(range(n))]),
        context_lens=i32([T]), cu_seqlens_q=i32([0, T]))


@GPU
def test_a_row_whose_norm_is_left_to_the_product(monkeypatch):
    """One row 4096 wide: 6144 outputs in the parts that 64 rows of weights want."""
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn(2, 1, 4096, generator=g, device="cuda")
    res, norm = (torch.randn(n, generator=g, device="cuda").bfloat16()
                 for n in ((1, 4096), (4096,)))
    w = (torch.randn(6144, 4096, generator=g, device="cuda") / 64).bfloat16()
    for steady, parts in ((True, 2), (False, 4)):
        h, new = ops.norm_ahead(x, res, norm, 1e-5, w, False, steady)
        assert isinstance(h, ops.Unnormed)
        y = ops.linear_parts(h, w, steady)
        assert y.shape == (parts, 1, 6144)
        if steady:
            rows, summed = ops.rmsnorm_residual(x, res, norm, 1e-5)
            assert torch.equal(new, summed)
            assert torch.equal(y, ops._hip.few_rows(rows, w, True, 2, 64))
    m, seen, real = _model(4096), [], ops.linear_parts

    def look(h, w, steady=False):
        y = real(h, w, steady)
        if w.shape[0] == 6144:
            seen.append((isinstance(h, ops.Unnormed), y.shape[0]))
        return y

    monkeypatch.setattr(ops, "linear_parts", look)
    m(*_parts(m, 1))
    assert seen == [(False, 2), (True, 2)]


class _Parts(LlamaMLP):
    def parts(self, x):
        return super().parts(2 * x)


@GPU
@pytest.mark.parametrize("how", ["class", "instance"])
def test_parts_of_its_own(how):
    """A user's own step is given the rows alone, as without an 8-bit cache."""
    m = _model()
    want = m(*_parts(m, 3))
    mlp = m.layers[0].mlp
    if how == "class":
        mlp.__class__ = _Parts
    else:
        mlp.parts = lambda x: LlamaMLP.parts(mlp, 2 * x)
    got = m(*_parts(m, 3))
    assert torch.isfinite(got).all() and not torch.equal(got, want)


@pytest.fixture
def forms(monkeypatch):
    """The forms that products of own kernels were asked in."""
    seen, real = [], ops._hip.own_product
    monkeypatch.setattr(ops._hip, "own_product",
                        lambda x, w, form: seen.append(form) or real(x, w, form))
    return seen


@GPU
@pytest.mark.parametrize("watched", [
    "", "layers.1", "layers.0.attn", "layers.1.attn.qkv_proj", "layers.0.attn.o_proj",
    "layers.0.mlp", "layers.1.mlp", "layers.0.mlp.gate_up", "layers.1.mlp.down"])
@pytest.mark.parametrize("T", [3, 300])
def test_whoever_watches(watched, T, forms):
    """Where a layer, a module or a product is watched, and the layer before it."""
    m, calls = _model(), []
    if watched:
        m.get_submodule(watched).register_forward_hook(lambda *a: calls.append(a[1]))
    m(*_parts(m, T))
    assert len(forms) >= 6 and all(f & 4 or f == 2 for f in forms)
    assert len(calls) == bool(watched) and all(
        isinstance(t, (torch.Tensor, tuple, AttnMetadata, type(None))) for c in calls for t in c)
    forms.clear()
    m(*_parts(m, T, eight=False))
    assert forms and not any(f & 4 for f in forms)


@GPU
def test_watched_experts(forms):
    m = _model(experts=2)
    m.layers[0].mlp.experts[1].register_forward_hook(lambda *a: None)
    m(*_parts(m, 300))
    # two layers' attention, one's experts
    assert len(forms) >= 6 and all(f & 4 or f == 2 for f in forms)


@GPU
def test_metadata_of_any_kind(forms):
    m = _model()
    m(*_parts(m, 3, kind=types.SimpleNamespace))
    assert len(forms) >= 6 and all(f & 4 or f == 2 for f in forms)


@GPU
@pytest.mark.parametrize("kind", [AttnMetadata, types.SimpleNamespace])
def test_layers_called_by_themselves(kind, forms):
    m = _model()
    ids, caches, meta = _parts(m, 3, kind=kind)
    m.layers[0](m.embed(ids), None, m.cos_sin, caches[0], meta)
    assert len(forms) >= 3 and all(f & 4 or f == 2 for f in forms)


class _NoCache(nn.Module):
    def forward(self, x, residual, cos_sin, kv_cache, meta):
        assert kv_cache is None
        return x, x if residual is None else residual


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=GPU)])
def test_a_first_layer_without_a_cache(device):
    """What replaces a layer need not have a cache."""
    m = _model(device=device)
    m.layers[0] = _NoCache()
    ids, caches, meta = _parts(m, 3, eight=False)
    assert torch.isfinite(m(ids, [None, caches[1]], meta)).all()
