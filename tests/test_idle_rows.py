"""Rows of a captured decode batch that no sequence fills."""
import pytest
import torch

from aurora_amd.engine.engine import EngineConfig, LLMEngine

pytestmark = pytest.mark.gpu


def test_idle_rows_hold_token_ids_whatever_the_pinned_memory_held():
    """The staging buffers may reuse pinned memory that held something else, an engine's
    ids of a larger vocabulary for one."""
    dirty = [torch.full((256,), 1 << 40, dtype=torch.int64).pin_memory() for _ in range(8)]
    del dirty
    eng = LLMEngine(EngineConfig(model="smoke-llama", kv_cache_pages=8, max_num_seqs=4))
    ids = eng._host_i64
    assert int(ids.min()) >= 0 and int(ids.max()) < eng.spec.vocab_size
