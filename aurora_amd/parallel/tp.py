"""Tensor-parallel linear layers (Megatron-style column/row split).

At tp_world_size()==1 these are plain bias-free linears; with TP the column
layer shards output features (heads / MLP intermediate) and the row layer
shards input features and all-reduces its partial outputs over RCCL/xGMI.
Weights are created pre-sharded (random init in this environment); the
loader shards checkpoints the same way.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules.module import (
    _global_backward_hooks,
    _global_backward_pre_hooks,
    _global_forward_hooks,
    _global_forward_pre_hooks,
)

from .. import ops
from . import dist as pdist

_CALL = nn.Module.__call__


def is_plain(module: nn.Module, kind: type) -> bool:
    """True where a call of ``module`` is ``kind.forward`` and nothing else: no hook, no
    other class's or its own forward. Only then may its work be done without the call."""
    own, cls = module.__dict__, type(module)
    return not (cls.forward is not kind.forward or cls.__call__ is not _CALL
                or "forward" in own or own["_forward_hooks"] or own["_forward_pre_hooks"]
                or own["_backward_hooks"] or own["_backward_pre_hooks"]
                or _global_forward_hooks or _global_forward_pre_hooks
                or _global_backward_hooks or _global_backward_pre_hooks)


def is_method(module: nn.Module, kind: type, name: str) -> bool:
    """True where ``module``'s method of a name is ``kind``'s, not its own or a subclass's."""
    return (name not in module.__dict__
            and getattr(type(module), name, None) is getattr(kind, name))


def told(m: nn.Module, x, kind: type, steady: bool, name: str = "") -> torch.Tensor:
    """``m(x)``, or its method ``name`` of x, which is told ``steady`` (see ``ops.linear``) where
    it is ``kind``'s, whoever watches it; one of a user's own is given what it always was."""
    step = getattr(m, name) if name else m
    if steady and is_method(m, kind, name or "forward"):
        return step(x, steady=True)
    return step(x)


class ColumnParallelLinear(nn.Module):
    """Y_local = X @ W_local^T, W_local = W[rank-th output shard]."""

    def __init__(self, in_features: int, out_features: int, dtype=None,
                 gather_output: bool = False, bias: bool = False):
        super().__init__()
        tp = pdist.tp_world_size()
        assert out_features % tp == 0, (out_features, tp)
        self.in_features = in_features
        self.out_features = out_features
        self.out_local = out_features // tp
        self.gather_output = gather_output
        self.weight = nn.Parameter(
            torch.empty(self.out_local, in_features, dtype=dtype), requires_grad=False
        )
        # output-feature bias shards with the weight rows (Qwen2-family
        # attention projections carry a bias; Llama/Mixtral do not)
        self.bias = nn.Parameter(
            torch.empty(self.out_local, dtype=dtype), requires_grad=False
        ) if bias else None

    def forward(self, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
        y = ops.linear(x, self.weight, steady)
        if self.bias is not None:
            y = y + self.bias
        if self.gather_output:
            y = pdist.tp_all_gather(y, dim=-1)
        return y


class RowParallelLinear(nn.Module):
    """Y = all_reduce(X_local @ W_local^T), W_local = W[rank-th input shard]."""

    def __init__(self, in_features: int, out_features: int, dtype=None):
        super().__init__()
        tp = pdist.tp_world_size()
        assert in_features % tp == 0, (in_features, tp)
        self.in_features = in_features
        self.in_local = in_features // tp
        self.out_features = out_features
        self.weight = nn.Parameter(
            torch.empty(out_features, self.in_local, dtype=dtype), requires_grad=False
        )

    def forward(self, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
        y = ops.linear(x, self.weight, steady)
        return pdist.tp_all_reduce(y)


class QKVParallelLinear(ColumnParallelLinear):
    """Fused QKV projection, head-sharded: local output is
    [q_heads_local*D | kv_heads_local*D | kv_heads_local*D]."""

    def __init__(self, hidden: int, n_heads: int, n_kv_heads: int, head_dim: int,
                 dtype=None, bias: bool = False):
        tp = pdist.tp_world_size()
        assert n_heads % tp == 0 and n_kv_heads % tp == 0, (n_heads, n_kv_heads, tp)
        self.n_heads_local = n_heads // tp
        self.n_kv_heads_local = n_kv_heads // tp
        self.head_dim = head_dim
        out = (n_heads + 2 * n_kv_heads) * head_dim
        super().__init__(hidden, out, dtype=dtype, bias=bias)

    def split_qkv(self, qkv: torch.Tensor):
        d = self.head_dim
        q = qkv[..., : self.n_heads_local * d]
        k = qkv[..., self.n_heads_local * d: (self.n_heads_local + self.n_kv_heads_local) * d]
        v = qkv[..., (self.n_heads_local + self.n_kv_heads_local) * d:]
        return q, k, v


class MergedColumnParallelLinear(ColumnParallelLinear):
    """gate|up fused projection: each half is sharded independently so the
    local output stays [gate_local | up_local] (silu_mul expects that)."""

    def __init__(self, hidden: int, intermediate: int, dtype=None):
        super().__init__(hidden, 2 * intermediate, dtype=dtype)
        self.intermediate_local = intermediate // pdist.tp_world_size()


def column_parts(m: nn.Module, x: torch.Tensor,
                 steady: bool = False) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """``m(x)`` of a column-parallel layer as a product possibly in parts
    (``ops.linear_parts``) and the bias still to be added."""
    if is_plain(m, ColumnParallelLinear) and not m.gather_output:
        return ops.linear_parts(x, m.weight, steady), m.bias
    return told(m, x, ColumnParallelLinear, steady), None


def column_weight(m: nn.Module, bias: bool) -> Optional[torch.Tensor]:
    """What ``column_parts`` (with ``bias``) or ``column_silu_mul`` multiplies by itself; None
    where it calls ``m``."""
    return m.weight if (is_plain(m, ColumnParallelLinear) and not m.gather_output
                        and (bias or m.bias is None)) else None


def row_parts(m: nn.Module, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
    """``m(x)`` of a row-parallel layer, possibly in parts where nothing is reduced."""
    if is_plain(m, RowParallelLinear) and pdist.tp_world_size() == 1:
        return ops.linear_parts(x, m.weight, steady)
    return row(m, x, steady)


def row(m: nn.Module, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
    """``m(x)`` of a row-parallel layer; ``steady`` as for ``ops.linear``."""
    return told(m, x, RowParallelLinear, steady)


def column_silu_mul(m: nn.Module, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
    """``silu_mul(m(x))`` of a merged gate and up layer, in one kernel where that is faster."""
    if is_plain(m, ColumnParallelLinear) and m.bias is None and not m.gather_output:
        return ops.linear_silu_mul(x, m.weight, steady)
    return ops.silu_mul(told(m, x, ColumnParallelLinear, steady))
