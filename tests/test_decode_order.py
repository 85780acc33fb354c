"""Decode attention over whole contexts, which start longest first."""
import pytest
import torch

from aurora_amd import ops
from test_decode_stretches import _case, _check, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["apart", "alike", "short", "one long", "powers"])
@pytest.mark.parametrize("B", [63, 64, 65, 128, 129, 256, 257])
def test_every_context_once(B, kind):
    """Around a wave's lanes, the numbers a lane holds and the batches that keep their order."""
    contexts = {"apart": [1 + 53 * i % 1471 for i in range(B)],
                "alike": [769 + i % 3 for i in range(B)],
                "short": [1 + i % 512 for i in range(B)],
                "one long": [1 + (1300 if i == B // 2 else i % 7) for i in range(B)],
                "powers": [(511, 512, 513, 1023, 1024, 1025)[i % 6] for i in range(B)]}[kind]
    q, k, v, bt, ctx = _case(contexts, 64, 32, 4, 64, torch.bfloat16)
    assert (8 * B) ** 2 // 16 >= bt.shape[1] * 64  # contexts stay whole
    out = torch.full_like(q, float("nan"))
    ops.paged_attention_decode(q, k, v, bt, ctx, 0.125, out=out)
    _check(out, _reference(q, k, v, bt, ctx, 0.125))
