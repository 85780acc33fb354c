"""Mixers and MLPs of layer-listed models that a user watches or replaces are called, and see
whole results; a few rows of others come in parts."""
import pytest
import torch

from aurora_amd import ops
from aurora_amd.engine.engine import EngineConfig, LLMEngine
from aurora_amd.engine.sampling_params import SamplingParams
from test_watched_modules import DEVICES, _same

DESIGNS = ["kikalix", "senotar", "gakupel", "fezuzen"]
PROMPTS = [list(range(30, 41)), [7], list(range(90, 103))]


def _logits(design, device, change=lambda model: None):
    """Of the last tokens of three prompts of 25 tokens."""
    size = "tiny" if device == "cpu" else "smoke"
    engine = LLMEngine(EngineConfig(model=f"{size}-{design}", device=device, kv_cache_pages=64,
                                    seed=3))
    change(engine.model)
    seen, whole = [], engine.model.compute_logits
    engine.model.compute_logits = lambda h: seen.append(whole(h)) or seen[-1]
    engine.generate(PROMPTS, SamplingParams(temperature=0.0, max_tokens=1, ignore_eos=True))
    return torch.cat([x[:, :512].float() for x in seen])


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("design", DESIGNS)
@pytest.mark.parametrize("kind", ["mixer", "mlp"])
def test_hooks(design, device, kind):
    seen = []

    def look(module, args, out):
        out = out if isinstance(out, torch.Tensor) else out.get("delta")
        seen.append(out)
        assert out is None or out.dim() == 2 and out.shape[0] == 25

    def watch(model):
        for layer in model.layers:
            if getattr(layer, kind) is not None:
                getattr(layer, kind).register_forward_hook(look)

    before = _logits(design, device)
    assert before.shape[0] == 3
    _same(_logits(design, device, watch), before)
    assert seen


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("design", DESIGNS)
@pytest.mark.parametrize("how", ["class", "instance"])
def test_forwards_of_their_own(design, device, how):
    """A mixer's forward that turns the sign does what a turned projection does."""
    def turn(model):
        model.layers[1].mixer.out_proj.data.neg_()  # exact

    def own(model):
        m = model.layers[1].mixer
        if how == "instance":
            m.forward = lambda *args, f=m.forward: -f(*args)
            return

        class Turned(type(m)):
            def forward(self, *args):
                return -super().forward(*args)

        m.__class__ = Turned

    want, plain = _logits(design, device, turn), _logits(design, device)
    assert (plain - want).norm() > 2 ** -5 * want.norm()
    _same(_logits(design, device, own), want)


@pytest.mark.gpu
def test_products_in_parts(monkeypatch):
    """Unwatched, the same rows do come in parts."""
    seen, parts = [], ops.linear_parts
    monkeypatch.setattr(ops, "linear_parts",
                        lambda x, w: seen.append(parts(x, w)) or seen[-1])
    _logits("kikalix", "cuda")
    assert any(y.dim() == 3 for y in seen)
