"""Batches put together in native code are those put together in Python."""
import numpy as np
import pytest
import torch

from aurora_amd import ops
from aurora_amd.engine.engine import EngineConfig, LLMEngine, Sequence
from aurora_amd.engine.sampling_params import SamplingParams
from aurora_amd.models.encoder import SentenceEncoder

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    return LLMEngine(EngineConfig(model="smoke-llama", page_size=64, kv_cache_pages=40,
                                  max_num_seqs=8))


def _sequence(engine, name, tokens, cached, ids=None):
    s = Sequence(name, ids or [(7 * i + len(name)) % 50 for i in range(tokens)],
                 SamplingParams())
    s.pages = engine.kv.alloc(-(-tokens // engine.kv.page_size))
    s.num_cached = cached
    return s


#: (tokens, cached, portion) of prompts; tokens of decoding sequences; page borders among them
STEPS = {"prompts": ([(64, 0, 64), (200, 63, 130), (65, 64, 1)], []),
         "decode": ([], [1, 64, 65, 130]),
         "mixed": ([(130, 128, 2), (1, 0, 1)], [64, 300])}


def _check(got, want):
    assert torch.equal(got[0], want[0]) and got[0].dtype == want[0].dtype
    a, b = vars(got[1]), vars(want[1])
    assert a.keys() == b.keys()
    for key in a:
        if isinstance(b[key], torch.Tensor):
            assert a[key].dtype == b[key].dtype and torch.equal(a[key], b[key]), key
            assert a[key].is_contiguous() and a[key].device == b[key].device, key
        else:
            assert a[key] == b[key], key


@pytest.mark.parametrize("step", STEPS)
def test_steps(engine, step, monkeypatch):
    prompts, decodes = STEPS[step]
    pre = [_sequence(engine, f"p{i}", t, c) for i, (t, c, _) in enumerate(prompts)]
    dec = [_sequence(engine, f"d{i}", t, t - 1) for i, t in enumerate(decodes)]
    chunks = [n for *_, n in prompts]
    assert engine._pack_batch(pre, chunks, dec) is not None
    got = engine._build_batch(pre, chunks, dec)
    monkeypatch.setattr(ops, "pack_batch", lambda *a: None)
    _check(got, engine._build_batch(pre, chunks, dec))
    for s in pre + dec:
        engine.kv.free(s.pages)


def test_other_integers(engine):
    """Ids that are no plain integers, and a token without a page, are left to Python."""
    s = _sequence(engine, "s", 3, 0, [np.int64(3), True, 5])
    assert engine._pack_batch([s], [3], []) is None
    assert engine._build_batch([s], [3], [])[0].tolist() == [3, 1, 5]
    bare = Sequence("bare", [1, 2], SamplingParams())
    with pytest.raises(IndexError):
        engine._build_batch([bare], [2], [])
    engine.kv.free(s.pages)


@pytest.mark.parametrize("texts", [[[4, 5], [], [6]], [[1]], [tuple(range(700)), [2, 3]],
                                   [[np.int32(4), 5], [7]]])
def test_texts(texts, monkeypatch):
    m = SentenceEncoder("bge-base", device="cuda")
    m.init_random(3)
    got = m.encode_ids(texts)
    monkeypatch.setattr(ops, "pack_texts", lambda *a: None)
    assert torch.equal(got, m.encode_ids([list(t) for t in texts]))
