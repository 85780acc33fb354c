"""Calls that the kernels have no form for are errors."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,res", [((9, 64), (9, 64)), ((1, 9, 64), (1, 9, 64)),
                                   ((1, 9, 64), (9, 64)), ((3, 9, 64), (3, 9, 64)),
                                   ((3, 9, 64), (1, 9, 64)), ((3, 9, 64), (9 * 64,))])
def test_norm_of_float32(x, res):
    with pytest.raises(RuntimeError):
        ops.rmsnorm_residual(torch.ones(x, device="cuda"),
                             torch.ones(res, device="cuda").bfloat16(),
                             torch.ones(64, device="cuda").bfloat16())
