"""Sentence-embedding encoder (BGE-class capability, aurora-native arch).

Replaces the reference's Weaviate text2vec-transformers sidecar (reference:
docker-compose.yaml:545) with an in-process encoder running entirely on the
existing gfx950 kernel set: bidirectional varlen attention
(ops.attention_prefill causal=False), RMSNorm, SiLU-MLP, RoPE positions,
mean-pool + L2 (ops.embed_pool).  Weights are random-init here (no network);
the architecture intentionally reuses the serving kernels so the embedder
adds zero new GPU surface.
"""
from __future__ import annotations

from typing import List

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import ops
from ..parallel.tp import is_method, is_plain
from .config import ModelSpec, get_spec


#: tokens of the longest text up to which attention rotates queries and keys itself. Every block
#: of 128 rows turns all keys of its text again: 54 texts of 512 tokens, 12 heads of 64, 138 us
#: and with the rotation apart 151; 8 of 2048 262 and 258; 3 of 8192 1445 and 1281.
TURNED_TOKENS = 1024


def _product(m: nn.Module, x: torch.Tensor, in_parts: bool = False) -> torch.Tensor:
    """``m(x)``, through the framework's products where nobody watches or replaced ``m``; with
    ``in_parts`` possibly in parts (``ops.linear_parts``)."""
    if is_plain(m, nn.Linear) and m.bias is None:
        return (ops.linear_parts if in_parts else ops.linear)(x, m.weight)
    return m(x)


class EncoderLayer(nn.Module):
    def __init__(self, spec: ModelSpec, dtype):
        super().__init__()
        h, d = spec.hidden_size, spec.head_dim
        self.n_heads = spec.n_heads
        self.head_dim = d
        self.scale = d ** -0.5
        self.norm1 = nn.Parameter(torch.ones(h, dtype=dtype), requires_grad=False)
        self.norm2 = nn.Parameter(torch.ones(h, dtype=dtype), requires_grad=False)
        self.qkv = nn.Linear(h, 3 * spec.n_heads * d, bias=False, dtype=dtype)
        self.o = nn.Linear(spec.n_heads * d, h, bias=False, dtype=dtype)
        self.gate_up = nn.Linear(h, 2 * spec.intermediate_size, bias=False, dtype=dtype)
        self.down = nn.Linear(spec.intermediate_size, h, bias=False, dtype=dtype)
        for p in self.parameters():
            p.requires_grad_(False)
        self.eps = spec.rms_eps

    def forward(self, x, cos_sin, positions, cu):
        x, delta = self.step(x, None, cos_sin, positions, cu)
        return x + delta

    def step(self, x, delta, cos_sin, positions, cu, in_order=False, in_parts=False):
        """The stream ``x``, to which ``delta`` (the layer before's result) is still to be
        added -> the stream and this layer's. ``in_order``: positions are the tokens' places
        in their texts; with ``in_parts`` the result may be in parts, as ``delta`` may be, which
        ``rmsnorm_residual`` adds up."""
        T = x.shape[0]
        if delta is None:
            h = ops.rmsnorm(x, self.norm1, self.eps)
        else:
            h, x = ops.rmsnorm_residual(delta, x, self.norm1, self.eps)
        qkv = _product(self.qkv, h).view(T, 3 * self.n_heads, self.head_dim)
        q, k, v = qkv.split(self.n_heads, dim=1)
        if in_order:
            o = ops.attention_prefill_turned(q, k, v, cos_sin, cu, self.scale, causal=False)
        else:
            if is_plain(self.qkv, nn.Linear):
                ops.rope_apply_(q, k, positions, cos_sin)
            else:  # what somebody else made may be kept by them
                q, k = ops.rope_apply(q.clone(), k.clone(), positions, cos_sin)
            o = ops.attention_prefill(q, k, v, cu, self.scale, causal=False)
        h, x = ops.rmsnorm_residual(_product(self.o, o.reshape(T, -1), True), x, self.norm2,
                                    self.eps)
        if is_plain(self.gate_up, nn.Linear) and self.gate_up.bias is None:
            act = ops.linear_silu_mul(h, self.gate_up.weight)
        else:
            act = ops.silu_mul(self.gate_up(h))
        return x, _product(self.down, act, in_parts)


class SentenceEncoder(nn.Module):
    def __init__(self, spec_name: str = "bge-base", dtype=torch.bfloat16, device="cpu"):
        super().__init__()
        spec = get_spec(spec_name)
        assert spec.is_encoder, spec_name
        self.spec = spec
        if device == "cpu":
            dtype = torch.float32
        self.embed = nn.Embedding(spec.vocab_size, spec.hidden_size, dtype=dtype)
        self.embed.weight.requires_grad_(False)
        self.layers = nn.ModuleList(
            [EncoderLayer(spec, dtype) for _ in range(spec.n_layers)])
        self.final_norm = nn.Parameter(torch.ones(spec.hidden_size, dtype=dtype),
                                       requires_grad=False)
        cs = ops.torch_ref.rope_cos_sin_cache(spec.head_dim, spec.max_position, 10000.0)
        self.register_buffer("cos_sin", cs, persistent=False)
        self.to(device)
        self.device_str = device

    @torch.inference_mode()
    def init_random(self, seed: int = 0) -> None:
        g = torch.Generator().manual_seed(seed)
        for p in self.parameters():
            if p.dim() >= 2:
                p.copy_((torch.randn(p.shape, generator=g) * p.shape[-1] ** -0.5).to(p.dtype))

    @torch.inference_mode()
    def encode_ids(self, batches: List[List[int]]) -> torch.Tensor:
        """[N, H] L2-normalized embeddings for N token-id lists."""
        dev = self.embed.weight.device
        maxp = self.spec.max_position
        batches = list(batches)
        packed = ops.pack_texts(batches, maxp, dev) if dev.type == "cuda" else None
        if packed is not None:
            ids, cu_t, pos_t = packed
        else:
            batches = [b[:maxp] if b else [0] for b in batches]
            flat = [t for b in batches for t in b]
            cu = [0]
            pos: List[int] = []
            for b in batches:
                cu.append(cu[-1] + len(b))
                pos.extend(range(len(b)))
            ids = torch.tensor(flat, dtype=torch.long, device=dev)
            cu_t = torch.tensor(cu, dtype=torch.int32, device=dev)
            pos_t = torch.tensor(pos, dtype=torch.int32, device=dev)
        in_order = maxp <= TURNED_TOKENS or max(map(len, batches), default=0) <= TURNED_TOKENS
        x = self.embed(ids)
        delta = None
        plain = [is_plain(layer, EncoderLayer) for layer in self.layers]
        # a step of a user's own knows nothing of parts: it neither is asked for them nor gets them
        known = [a and is_method(layer, EncoderLayer, "step")
                 for a, layer in zip(plain, self.layers)] + [True]
        for i, layer in enumerate(self.layers):
            if known[i]:
                x, delta = layer.step(x, delta, self.cos_sin, pos_t, cu_t, in_order, known[i + 1])
            elif plain[i]:
                x, delta = layer.step(x, delta, self.cos_sin, pos_t, cu_t, in_order)
            else:  # somebody watches it or has replaced it
                x, delta = x if delta is None else x + delta, None
                x = layer(x, self.cos_sin, pos_t, cu_t)
        if delta is None:
            x = ops.rmsnorm(x, self.final_norm, self.spec.rms_eps)
        else:
            x = ops.rmsnorm_residual(delta, x, self.final_norm, self.spec.rms_eps)[0]
        return ops.embed_pool(x, cu_t)
