"""A step of one row, whose norms are left to the products that read them, where those are a
user's own or watched."""
import types

import pytest
import torch

from aurora_amd import ops
from aurora_amd.models.llama import LlamaAttention, LlamaMLP
from test_watched_modules import _model, _same, _step

pytestmark = pytest.mark.gpu


@pytest.fixture
def left(monkeypatch):
    """The norms that were left to a product."""
    seen, ahead = [], ops.norm_ahead

    def look(*args):
        rows, new = ahead(*args)
        seen.append(isinstance(rows, ops.Unnormed))
        return rows, new

    monkeypatch.setattr(ops, "norm_ahead", look)
    return seen


def test_bits_of_separate_norms(left, monkeypatch):
    m = _model("smoke-llama", "cuda")
    got = _step(m, 1)
    # the first layer's first norm reads the embedding, the model's last the last layer's product
    assert sum(left) == len(left) == 2 * len(m.layers) - 1
    monkeypatch.setattr(ops, "norm_ahead", lambda x, res, w, eps, *_: ops.rmsnorm_residual(
        x, res, w, eps))
    assert torch.equal(_step(m, 1), got)


class _Heads(LlamaAttention):
    def _heads(self, x, *args):
        assert isinstance(x, torch.Tensor) and x.dim() == 2
        return super()._heads(2 * x, *args)


class _Parts(LlamaMLP):
    def parts(self, x):
        assert isinstance(x, torch.Tensor) and x.dim() == 2
        return super().parts(2 * x)


@pytest.mark.parametrize("how", ["class", "instance"])
@pytest.mark.parametrize("name,cls", [("attn", _Heads), ("mlp", _Parts)])
def test_steps_of_its_own(left, name, cls, how):
    """A step between the norm and the product sees the norm's rows, as with many rows."""
    plain, m = _model("tiny-llama", "cuda"), _model("tiny-llama", "cuda")
    own, step = m.layers[1].get_submodule(name), "_heads" if name == "attn" else "parts"
    if how == "class":
        own.__class__ = cls
    else:
        setattr(own, step, types.MethodType(
            lambda self, x, *args, f=getattr(own, step): f(2 * x, *args), own))
    read = {"attn": "attn.qkv_proj", "mlp": "mlp.gate_up"}[name]
    plain.layers[1].get_submodule(read).weight.data.mul_(2)  # exact
    want = _step(plain, 1)
    count = sum(left)
    got = _step(m, 1)
    assert sum(left) == 2 * count - 1  # the others are left to their products
    _same(got, want)
