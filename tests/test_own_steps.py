"""Steps that a user's own class has in a framework's place are called as they always were."""
import pytest
import torch

from aurora_amd.models.config import ModelSpec
from aurora_amd.models.encoder import EncoderLayer, SentenceEncoder
from aurora_amd.models.llama import MoEMLP
from aurora_amd.parallel import ep

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


class _Step(EncoderLayer):
    def step(self, x, delta, cos_sin, positions, cu, in_order=False):
        assert delta is None or delta.shape == x.shape
        x, delta = super().step(x, delta, cos_sin, positions, cu, in_order)
        return x, delta * 2


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("how", ["class", "instance"])
@pytest.mark.parametrize("at", [0, 5, 11])
def test_encoder_layer(device, how, at):
    """It takes no word about parts and gets none; nobody else's results are other ones."""
    e = SentenceEncoder("bge-base", dtype=torch.bfloat16 if device == "cuda" else torch.float32,
                        device=device)
    e.init_random(0)
    texts = [[5, 6, 7, 8], list(range(40, 240))]
    with torch.inference_mode():
        plain = e.encode_ids(texts)
        layer = e.layers[at]
        if how == "class":
            layer.__class__ = _Step
        else:
            layer.step = lambda *a: _Step.step(_as(layer), *a)
        own = e.encode_ids(texts)
        # the same said by a forward of its own
        layer.__dict__.pop("step", None)
        layer.__class__ = EncoderLayer
        layer.forward = lambda x, *a: sum(_twice(layer.step(x, None, *a)))
        want = e.encode_ids(texts)
    assert not torch.equal(own, plain)
    # 16 bits: a row rounds the other way at some places of some layers
    tol = 1e-5 if device == "cpu" else 2 ** -8 * e.spec.n_layers
    assert (own - want).float().norm() <= tol * want.float().norm()


def _twice(made):
    return made[0], made[1] * 2


def _as(layer):
    """The layer as one of the class above."""
    other = _Step.__new__(_Step)
    other.__dict__ = {k: v for k, v in layer.__dict__.items() if k != "step"}
    return other


class _Experts(MoEMLP):
    def _local_expert_fn(self, xp, local_sel):
        return xp * 2


@pytest.mark.parametrize("kind", [_Experts, MoEMLP])
@pytest.mark.parametrize("steady", [False, True])
def test_local_experts(kind, steady, monkeypatch):
    spec = ModelSpec(name="t", vocab_size=64, hidden_size=64, n_layers=1, n_heads=1, n_kv_heads=1,
                     head_dim=64, intermediate_size=64, n_experts=4)
    monkeypatch.setattr(ep, "ep_size", lambda: 2)
    monkeypatch.setattr(ep, "ep_moe_forward", lambda x, w, sel, n, fn: fn(x, sel[:, 0] % 2))
    m = kind(spec, torch.float32)
    for p in m.parameters():
        torch.nn.init.normal_(p, std=0.1, generator=torch.Generator().manual_seed(0))
    x = torch.randn(5, 64, generator=torch.Generator().manual_seed(1))
    y = m(x, steady=True) if steady else m(x)
    assert torch.equal(y, x * 2) == (kind is _Experts) and torch.equal(y, m(x))
