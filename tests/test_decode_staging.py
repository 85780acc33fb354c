"""A captured decode step's inputs, put together in native code and in Python."""
import types

import pytest
import torch

from aurora_amd import ops
from aurora_amd.engine.engine import LLMEngine, Sequence
from aurora_amd.engine.sampling_params import SamplingParams

PAGE, WIDTH, SCRATCH = 16, 5, 9


def _sequence(tokens, pages, slot=-1):
    s = Sequence("s", list(range(100, 100 + tokens)), SamplingParams())
    s.pages, s.state_slot = list(pages), slot
    return s


class _Staging:
    """A bucket's buffers, and an engine as far as staging in Python looks at it."""

    def __init__(self, bucket):
        self.ids = torch.zeros(8, dtype=torch.int64)
        self.host = torch.zeros(bucket + ((4 + WIDTH) * bucket + 1) // 2, dtype=torch.int64)
        self.inputs, self.keys = self.host.clone(), torch.full((bucket, 3), -1)
        rest = self.host[bucket:].view(torch.int32)
        self.parts = (self.host[:bucket], rest[:4 * bucket].view(4, bucket),
                      rest[4 * bucket:(4 + WIDTH) * bucket].view(bucket, WIDTH))
        self.parts[2].fill_(SCRATCH)
        self.engine = types.SimpleNamespace(
            _host_i64=self.ids, _scratch_page=SCRATCH, _scratch_slot=SCRATCH * PAGE,
            kv=types.SimpleNamespace(page_size=PAGE))
        self.engine._slot = types.MethodType(LLMEngine._slot, self.engine)

    def native(self, seqs):
        return ops.stage_decode(seqs, self.ids, self.host, self.keys, self.inputs, WIDTH, PAGE,
                                SCRATCH, SCRATCH * PAGE)

    def python(self, seqs):
        LLMEngine._stage_decode(self.engine, seqs, self.parts, self.keys)
        self.inputs.copy_(self.host)


@pytest.mark.parametrize("bucket", [1, 4, 8])
def test_as_in_python(bucket):
    """Steps of a batch that grows, gains pages, loses and swaps sequences; longer tables than
    a row holds; every step's buffer is the one put together in Python."""
    a, b = _Staging(bucket), _Staging(bucket)
    seqs = [_sequence(16 * k + 1 + k, range(k, 2 * k + 2), slot=k - 1) for k in range(bucket)]
    steps = [seqs[:1], seqs, seqs, seqs[::-1], seqs[1:] or seqs, [_sequence(70, range(7, 14))]]
    for i, step in enumerate(steps):
        for s in step:
            s.token_ids.append(1000 + i)
            if s.num_tokens > len(s.pages) * PAGE:
                s.pages.append(30 + i)
        if i == 3:  # freed, and other pages of the same number
            seqs[0].pages = [p + 40 for p in seqs[0].pages]
            seqs[0].page_gen += 1
        assert a.native(step)
        b.python(step)
        assert torch.equal(a.inputs, b.inputs) and torch.equal(a.ids, b.ids)


@pytest.mark.parametrize("what", ["tuple", "float", "numpy", "large page", "large slot", "empty"])
def test_left_to_python(what):
    """What native code does not take; a later plain step finds nothing stale."""
    import numpy as np
    a, b = _Staging(4), _Staging(4)
    good = _sequence(20, [3, 4])
    assert a.native([good, good])
    b.python([good, good])
    odd = _sequence(20, [3, 4])
    if what == "tuple":
        odd.token_ids = tuple(odd.token_ids)
    elif what == "float":
        odd.token_ids[-1] = 3.0
    elif what == "numpy":
        odd.pages = [np.int64(3), np.int64(4)]
    elif what == "large page":
        odd.pages[0] = 1 << 40
    elif what == "large slot":
        odd.pages[1] = 1 << 30
    else:
        odd.token_ids = []
    assert not a.native([good, odd])
    assert a.native([good])
    b.python([good])
    assert torch.equal(a.inputs, b.inputs)


@pytest.mark.parametrize("what", ["large page", "large slot", "empty"])
def test_refused_by_both(what):
    """A sequence that staging in Python refuses as well leaves no row that is taken for staged."""
    a, b = _Staging(4), _Staging(4)
    good, other, odd = (_sequence(20, pages) for pages in ([3, 4], [5, 6], [7, 8]))
    assert a.native([good, other])
    if what == "large page":
        odd.pages[0] = 1 << 40
    elif what == "large slot":
        odd.pages[1] = 1 << 30
    else:
        odd.token_ids = []
    assert not a.native([odd, other])
    with pytest.raises((RuntimeError, ValueError, IndexError, OverflowError)):
        a.python([odd, other])
    assert a.native([good, other])
    b.python([good, other])
    assert torch.equal(a.inputs, b.inputs)


@pytest.mark.gpu
def test_rows_on_the_device():
    assert ops.pack_rows([3, -1, 1 << 40], "cuda").tolist() == [3, -1, 1 << 40]
    assert ops.pack_rows([], "cuda") is None and ops.pack_rows([True], "cuda") is None
