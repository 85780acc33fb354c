"""Llama-3 / Qwen2-family decoder (GQA, RoPE, SiLU-MLP, optional QKV bias)
built on the aurora_amd op set.

Every hot op routes through aurora_amd.ops (HIP/CDNA4 kernels on GPU, fp32
torch reference on CPU), plain projections through ops.linear.
The forward is engine-shaped: packed varlen tokens + paged KV metadata, no
[B, S] padding anywhere.

Replaces the reference's rented chat models (reference:
server/chat/backend/agent/llm.py:39-67, providers/) with an in-process
model the engine steps directly.
"""
from __future__ import annotations

from copy import copy
from dataclasses import dataclass
from functools import partial
from typing import List, Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.utils.dlpack import from_dlpack, to_dlpack

from .. import ops
from ..parallel import dist as pdist
from ..parallel.tp import (
    ColumnParallelLinear,
    MergedColumnParallelLinear,
    QKVParallelLinear,
    RowParallelLinear,
    column_parts,
    column_silu_mul,
    column_weight,
    is_method,
    is_plain,
    row,
    row_parts,
    told,
)
from .config import ModelSpec


@dataclass
class AttnMetadata:
    """Per-step attention metadata shared by all layers.

    mode "prefill": q tokens are packed varlen chunks (cu_seqlens_q); their
    K/V have already been assigned cache slots via slot_mapping and the
    kernel attends against the paged cache (covers fresh and append prefill).
    mode "decode": one q token per sequence.
    """

    mode: str  # "prefill" | "decode" | "mixed"
    positions: torch.Tensor  # [T] int32 absolute positions
    slot_mapping: torch.Tensor  # [T] int32 cache slots for the new K/V
    block_tables: torch.Tensor  # [num_seqs, max_pages] int32
    context_lens: torch.Tensor  # [num_seqs] int32 (incl. new tokens)
    cu_seqlens_q: Optional[torch.Tensor] = None  # [num_seqs+1] int32, prefill only
    # mixed mode: tokens are [prefill chunks..., decode tokens]; the fields
    # above describe the prefill part, the ones below the decode part
    num_prefill_tokens: int = 0
    dec_block_tables: Optional[torch.Tensor] = None
    dec_context_lens: Optional[torch.Tensor] = None
    # models with recurrent layers: the state tensors of every recurrent run
    # and each sequence's slot in them (-1: an idle row, nothing is stored)
    states: Optional[List[Tuple[torch.Tensor, ...]]] = None
    state_slots: Optional[torch.Tensor] = None
    dec_state_slots: Optional[torch.Tensor] = None
    cu_host: Optional[List[int]] = None  # cu_seqlens_q without a device read
    ctx_host: Optional[List[int]] = None  # context_lens of the prompt portions
    marks: Optional[torch.Tensor] = None  # ``ops.decode_marks`` of the single tokens
    # decode: every row is the last token of a sequence that no other row belongs to, at the
    # position before its context's end and in the slot that its table names for it. (Rows that
    # nobody reads may share a page that is nobody's, as a captured batch's idle rows do)
    last_tokens: bool = False
    # prompts that fill an 8-bit cache: the products' sums keep their order (``ops.linear``).
    # The model finds it out once a step, layers called by themselves each for itself
    steady: Optional[bool] = None

    def segments(self, T: int) -> List[ops.Segment]:
        """The step's prompt portions and its single-token rows, each with its
        own tables, for layers that treat the two regimes apart."""
        Tp = {"prefill": T, "decode": 0}.get(self.mode, self.num_prefill_tokens)
        out = []
        if Tp:
            cu = self.cu_seqlens_q
            out.append(ops.Segment(
                rows=slice(0, Tp), block_tables=self.block_tables,
                context_lens=self.context_lens,
                starts=self.context_lens - (cu[1:] - cu[:-1]),
                state_slots=self.state_slots, cu=cu,
                cu_host=self.cu_host or cu.tolist(),
                ctx_host=self.ctx_host or self.context_lens.tolist()))
        if T > Tp:
            mixed = self.mode == "mixed"
            out.append(ops.Segment(
                rows=slice(Tp, T),
                block_tables=self.dec_block_tables if mixed else self.block_tables,
                context_lens=self.dec_context_lens if mixed else self.context_lens,
                starts=self.positions[Tp:],
                state_slots=self.dec_state_slots if mixed else self.state_slots))
        return out


def _eight_bits(kv_cache) -> bool:
    try:
        return kv_cache[0].element_size() == 1
    except (TypeError, LookupError, AttributeError):
        return False  # what a layer that replaced another may have


def _steady(meta, kv_cache) -> bool:
    """``AttnMetadata.steady`` of metadata of any kind."""
    known = getattr(meta, "steady", None)
    if known is None:
        return getattr(meta, "mode", "decode") != "decode" and _eight_bits(kv_cache)
    return known


class LlamaAttention(nn.Module):
    def __init__(self, spec: ModelSpec, dtype):
        super().__init__()
        self.spec = spec
        tp = pdist.tp_world_size()
        self.n_heads = spec.n_heads // tp
        self.n_kv_heads = spec.n_kv_heads // tp
        self.head_dim = spec.head_dim
        self.scale = spec.head_dim ** -0.5
        self.qkv_proj = QKVParallelLinear(
            spec.hidden_size, spec.n_heads, spec.n_kv_heads, spec.head_dim,
            dtype=dtype, bias=spec.qkv_bias
        )
        self.o_proj = RowParallelLinear(spec.q_size, spec.hidden_size, dtype=dtype)

    def forward(
        self,
        x: torch.Tensor,  # [T, H]
        cos_sin: torch.Tensor,
        kv_cache: Tuple[torch.Tensor, torch.Tensor],
        meta: AttnMetadata,
    ) -> torch.Tensor:
        return row(self.o_proj, self._heads(x, cos_sin, kv_cache, meta), _steady(meta, kv_cache))

    def parts(self, x, cos_sin, kv_cache, meta) -> torch.Tensor:
        """As ``forward``, possibly in parts (``ops.linear_parts``)."""
        return row_parts(self.o_proj, self._heads(x, cos_sin, kv_cache, meta),
                         _steady(meta, kv_cache))

    def _heads(self, x, cos_sin, kv_cache, meta) -> torch.Tensor:
        """The heads' results side by side, [T, heads * width]."""
        T = x.shape[0]
        qkv, bias = column_parts(self.qkv_proj, x, _steady(meta, kv_cache))
        k_cache, v_cache = kv_cache
        if meta.mode == "decode" and getattr(meta, "last_tokens", False):
            o = ops.fresh_attention_decode(
                qkv, bias, meta.positions, meta.slot_mapping, cos_sin, k_cache, v_cache,
                meta.block_tables, meta.context_lens, self.n_heads, self.scale,
                getattr(meta, "marks", None))
            return o.reshape(T, self.n_heads * self.head_dim)
        # fused split + bias + RoPE + paged K/V scatter (one kernel on GPU)
        q = ops.fused_rope_kv_write(qkv, meta.positions, meta.slot_mapping,
                                    cos_sin, k_cache, v_cache,
                                    self.n_heads, self.n_kv_heads, bias)
        if meta.mode == "prefill":
            o = ops.attention_prefill_paged(
                q, k_cache, v_cache, meta.block_tables,
                meta.cu_seqlens_q, meta.context_lens, self.scale,
            )
        elif meta.mode == "decode":
            o = ops.paged_attention_decode(
                q, k_cache, v_cache, meta.block_tables, meta.context_lens, self.scale,
                marks=getattr(meta, "marks", None),
            )
        else:  # mixed: prefill chunks + decode tokens in one forward — the
            # projections/norms run on the whole packed batch (bigger GEMMs),
            # attention splits per regime
            Tp = meta.num_prefill_tokens
            o = torch.empty_like(q)
            if Tp:
                ops.attention_prefill_paged(
                    q[:Tp], k_cache, v_cache, meta.block_tables,
                    meta.cu_seqlens_q, meta.context_lens, self.scale, out=o[:Tp],
                )
            if T > Tp:
                ops.paged_attention_decode(
                    q[Tp:], k_cache, v_cache, meta.dec_block_tables,
                    meta.dec_context_lens, self.scale, out=o[Tp:],
                    marks=getattr(meta, "marks", None),
                )
        return o.reshape(T, self.n_heads * self.head_dim)


class LlamaMLP(nn.Module):
    def __init__(self, spec: ModelSpec, dtype):
        super().__init__()
        self.gate_up = MergedColumnParallelLinear(spec.hidden_size, spec.intermediate_size, dtype=dtype)
        self.down = RowParallelLinear(spec.intermediate_size, spec.hidden_size, dtype=dtype)

    def forward(self, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
        return row(self.down, column_silu_mul(self.gate_up, x, steady), steady)

    def parts(self, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
        """As ``forward``, possibly in parts (``ops.linear_parts``)."""
        return row_parts(self.down, column_silu_mul(self.gate_up, x, steady), steady)


class _FullWidthMLP(nn.Module):
    """Unsharded SiLU MLP for expert-parallel mode: the whole expert lives
    on its owner rank (no intra-expert TP, no per-expert all-reduce)."""

    def __init__(self, spec: ModelSpec, dtype):
        super().__init__()
        self.gate_up = nn.Parameter(torch.empty(
            2 * spec.intermediate_size, spec.hidden_size, dtype=dtype),
            requires_grad=False)
        self.down = nn.Parameter(torch.empty(
            spec.hidden_size, spec.intermediate_size, dtype=dtype),
            requires_grad=False)

    def forward(self, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
        return ops.linear(ops.linear_silu_mul(x, self.gate_up, steady), self.down, steady)


def _are_slices(whole: Optional[torch.Tensor], weights: List[torch.Tensor]) -> bool:
    """True where ``weights`` are ``whole[0]``, ``whole[1]`` and so on themselves."""
    if whole is None or whole.is_meta:
        return False
    at, step, shape = whole.data_ptr(), whole.stride(0) * whole.element_size(), whole.shape[1:]
    return all(w.data_ptr() == at + i * step and w.shape == shape and w.dtype == whole.dtype
               and w.is_contiguous() for i, w in enumerate(weights))


def _apart(x: torch.Tensor) -> torch.Tensor:
    """The same memory with a storage of its own: whoever saves ``x`` saves no more, and
    does not find it to be a part of something."""
    return x if x.is_meta else from_dlpack(to_dlpack(x))


class MoEMLP(nn.Module):
    """Mixtral-style sparse MoE block (top-k routing over dense experts).

    Experts are TP-sharded like the dense MLP (each expert's gate_up column-
    sharded, down row-sharded) so the expert compute stays local and the
    row-parallel all-reduce doubles as the TP combine.  On the GPU tokens are
    sorted by expert on the device and run through grouped products; elsewhere
    dispatch is a host-side gather for prompts, a batched product for small batches.
    """

    def __init__(self, spec: ModelSpec, dtype):
        super().__init__()
        from ..parallel import ep as pep
        self.n_experts = spec.n_experts
        self.top_k = spec.experts_per_token
        self.router = nn.Linear(spec.hidden_size, spec.n_experts, bias=False, dtype=dtype)
        self.router.weight.requires_grad_(False)
        self.ep_size = pep.ep_size()
        if self.ep_size > 1:
            # expert parallelism (AURORA_EP=1): this rank owns
            # n_experts/ep FULL-width experts; tokens travel to their
            # experts over all-to-all instead of sharding each expert
            assert spec.n_experts % self.ep_size == 0
            self.e_local = spec.n_experts // self.ep_size
            self.experts = nn.ModuleList(
                [_FullWidthMLP(spec, dtype) for _ in range(self.e_local)])
        else:
            self.experts = nn.ModuleList(
                [LlamaMLP(spec, dtype) for _ in range(spec.n_experts)]
            )
        self._w_gu = None  # all experts' weights in one tensor each, in whose memory the
        self._w_dn = None  # experts' own lie
        if self.ep_size == 1:
            gu, dn = self.experts[0].gate_up.weight, self.experts[0].down.weight
            self._share(gu.new_empty((self.n_experts, *gu.shape)),
                        dn.new_empty((self.n_experts, *dn.shape)))

    def _share(self, w_gu: torch.Tensor, w_dn: torch.Tensor) -> None:
        for e, ex in enumerate(self.experts):
            ex.gate_up.weight.data, ex.down.weight.data = _apart(w_gu[e]), _apart(w_dn[e])
        self._w_gu, self._w_dn = w_gu, w_dn

    def _apply(self, fn, recurse: bool = True):
        self._w_gu = self._w_dn = None  # a move leaves every expert's weights apart
        return super()._apply(fn, recurse)

    def _stacked(self) -> Tuple[torch.Tensor, torch.Tensor]:
        """All experts' weights, put together anew if one has got another storage
        (``load_state_dict(assign=True)``, a copy of the module, ``weight.data``)."""
        gu = [ex.gate_up.weight for ex in self.experts]
        dn = [ex.down.weight for ex in self.experts]
        if not (_are_slices(self._w_gu, gu) and _are_slices(self._w_dn, dn)):
            with torch.inference_mode(gu[0].is_inference()):
                self._share(torch.stack([w.data for w in gu]),
                            torch.stack([w.data for w in dn]))
        return self._w_gu, self._w_dn

    def _experts_plain(self) -> bool:
        """True where router and experts are what this class made them and nobody watches."""
        return is_plain(self.router, nn.Linear) and all(
            is_plain(ex, LlamaMLP) and is_plain(ex.gate_up, ColumnParallelLinear)
            and is_plain(ex.down, RowParallelLinear) for ex in self.experts)

    def _local_expert_fn(self, xp: torch.Tensor, local_sel: torch.Tensor,
                         steady: bool = False) -> torch.Tensor:
        y = torch.empty_like(xp)
        for le in range(self.e_local):
            m = (local_sel == le)
            if m.any():
                y[m] = told(self.experts[le], xp[m], _FullWidthMLP, steady)
        return y

    def forward(self, x: torch.Tensor, steady: bool = False) -> torch.Tensor:
        T, H = x.shape
        if (self.ep_size == 1 and self._experts_plain()
                and ops.has_moe_grouped(x, self.router.weight)):
            out = ops.moe_silu_glu(x, self.router.weight, self.top_k, *self._stacked())
            return pdist.tp_all_reduce(out) if pdist.tp_world_size() > 1 else out
        logits = self.router(x).float()  # [T, E]
        weights, sel = logits.topk(self.top_k, dim=-1)
        weights = weights.softmax(-1).to(x.dtype)  # [T, k]
        if self.ep_size > 1:
            from ..parallel import ep as pep
            local = self._local_expert_fn
            if steady and is_method(self, MoEMLP, "_local_expert_fn"):
                local = partial(local, steady=True)
            return pep.ep_moe_forward(x, weights, sel, self.n_experts, local)
        if T <= 256:
            return self._forward_batched(x, weights, sel)
        # prefill: per-expert token batches are large, so plain per-expert
        # GEMMs are efficient and avoid the capacity buffer
        out = torch.zeros_like(x)
        for e in range(self.n_experts):
            tok, slot = (sel == e).nonzero(as_tuple=True)
            if tok.numel() == 0:
                continue
            y = told(self.experts[e], x[tok], LlamaMLP, steady)
            out.index_add_(0, tok, y * weights[tok, slot, None])
        return out

    def _forward_batched(self, x: torch.Tensor, weights: torch.Tensor,
                         sel: torch.Tensor) -> torch.Tensor:
        """Small batches without the router kernel: tokens sorted by expert and packed for
        one product per expert that was chosen, or without the extension in a buffer of
        fixed capacity for batched products over all experts. Static shapes, nothing read
        back."""
        T, H = x.shape
        E, k = self.n_experts, self.top_k
        flat = sel.reshape(-1)  # [T*k]
        order = flat.argsort(stable=True)  # tokens grouped by expert
        tok_of = order // k  # token index of each sorted assignment
        # histogram via scatter_add (bincount host-syncs -> not capturable)
        counts = torch.zeros(E, dtype=torch.long, device=x.device).scatter_add_(
            0, flat, torch.ones_like(flat))
        starts = torch.cumsum(counts, 0) - counts
        w_gu, w_dn = self._stacked()
        wflat = weights.reshape(-1)[order].unsqueeze(1).to(x.dtype)
        out = torch.zeros_like(x)
        if ops.has_moe_grouped(x):
            st, ct = starts.to(torch.int32), counts.to(torch.int32)
            act = ops.silu_mul(ops.moe_grouped_gemm(x[tok_of], w_gu, st, ct))  # [T*k, I']
            out.index_add_(0, tok_of, ops.moe_grouped_gemm(act, w_dn, st, ct) * wflat)
            return pdist.tp_all_reduce(out) if pdist.tp_world_size() > 1 else out
        C = T
        rank = torch.arange(T * k, device=x.device) - starts[flat[order]]
        slot_idx = flat[order] * C + rank  # rank < C always
        xe = x.new_zeros(E * C, H)
        xe[slot_idx] = x[tok_of]
        xe = xe.view(E, C, H)
        gu = torch.bmm(xe, w_gu.transpose(1, 2).contiguous())  # [E, C, 2I']
        act = ops.silu_mul(gu.reshape(E * C, -1)).view(E, C, -1)
        ye = torch.bmm(act, w_dn.transpose(1, 2).contiguous()).view(E * C, H)
        out.index_add_(0, tok_of, ye[slot_idx] * wflat)
        return pdist.tp_all_reduce(out) if pdist.tp_world_size() > 1 else out


class LlamaDecoderLayer(nn.Module):
    def __init__(self, spec: ModelSpec, dtype):
        super().__init__()
        self.input_norm = nn.Parameter(torch.empty(spec.hidden_size, dtype=dtype), requires_grad=False)
        self.post_attn_norm = nn.Parameter(torch.empty(spec.hidden_size, dtype=dtype), requires_grad=False)
        self.eps = spec.rms_eps
        self.attn = LlamaAttention(spec, dtype)
        self.mlp = MoEMLP(spec, dtype) if spec.n_experts > 0 else LlamaMLP(spec, dtype)

    def forward(self, x, residual, cos_sin, kv_cache, meta):
        return self.step(x, residual, cos_sin, kv_cache, meta, False)

    def step(self, x, residual, cos_sin, kv_cache, meta, in_parts: bool):
        """As ``forward``; with ``in_parts`` the result may be in parts, which
        ``rmsnorm_residual`` adds up, and so may ``x``."""
        steady = _steady(meta, kv_cache)
        if residual is None:
            residual = x
            h = ops.rmsnorm(x, self.input_norm, self.eps)
        else:
            h, residual = ops.norm_ahead(x, residual, self.input_norm, self.eps,
                                         self._reader("attn", x), False, steady)
        attn = self.attn.parts if is_plain(self.attn, LlamaAttention) else self.attn
        a = attn(h, cos_sin, kv_cache, meta)
        h, residual = ops.norm_ahead(a, residual, self.post_attn_norm, self.eps,
                                     self._reader("mlp", a) if in_parts else None, True, steady)
        if in_parts and is_plain(self.mlp, LlamaMLP):
            return told(self.mlp, h, LlamaMLP, steady, "parts"), residual
        kind = MoEMLP if isinstance(self.mlp, MoEMLP) else LlamaMLP
        return told(self.mlp, h, kind, steady), residual

    def _reader(self, what: str, x: torch.Tensor) -> Optional[torch.Tensor]:
        """The weight whose product alone reads the norm before ``what``, if x, the norm's
        input, is a single row in parts and nobody watches the product."""
        if x.dim() != 3 or x.shape[1] != 1:
            return None
        module, kind, inner = ((self.attn, LlamaAttention, ("parts", "_heads")) if what == "attn"
                               else (self.mlp, LlamaMLP, ("parts",)))
        # (a subclass's own steps are given rows, as they always were)
        if not is_plain(module, kind) or any(
                getattr(getattr(module, n), "__func__", None) is not getattr(kind, n)
                for n in inner):
            return None
        return (column_weight(module.qkv_proj, True) if kind is LlamaAttention
                else column_weight(module.gate_up, False))


class LlamaForCausalLM(nn.Module):
    def __init__(self, spec: ModelSpec, dtype=torch.bfloat16, device=None):
        super().__init__()
        self.spec = spec
        self.dtype = dtype
        self.embed = nn.Embedding(spec.vocab_size, spec.hidden_size, dtype=dtype)
        self.embed.weight.requires_grad_(False)
        self.layers = nn.ModuleList(
            [LlamaDecoderLayer(spec, dtype) for _ in range(spec.n_layers)]
        )
        self.final_norm = nn.Parameter(torch.empty(spec.hidden_size, dtype=dtype), requires_grad=False)
        if spec.tie_embeddings:
            self.lm_head = None
        else:
            self.lm_head = nn.Linear(spec.hidden_size, spec.vocab_size, bias=False, dtype=dtype)
            self.lm_head.weight.requires_grad_(False)
        cos_sin = ops.torch_ref.rope_cos_sin_cache(
            spec.head_dim, spec.max_position, spec.rope_theta, dtype=torch.float32
        )
        self.register_buffer("cos_sin", cos_sin, persistent=False)
        if device is not None:
            self.to(device)

    def kv_layout(self) -> List[Tuple[int, int, int]]:
        """(kv heads, key width, value width) of every layer's paged cache."""
        s = self.spec
        heads = max(s.n_kv_heads // pdist.tp_world_size(), 1)
        return [(heads, s.head_dim, s.head_dim)] * s.n_layers

    def state_layout(self) -> List[tuple]:
        """No layer carries a recurrent state."""
        return []

    @torch.inference_mode()
    def forward(
        self,
        input_ids: torch.Tensor,  # [T]
        kv_caches: List[Tuple[torch.Tensor, torch.Tensor]],
        meta: AttnMetadata,
    ) -> torch.Tensor:
        x = self.embed(input_ids)
        residual = None
        if isinstance(meta, AttnMetadata):  # of another kind every layer makes its own marks
            tables = {"decode": meta.block_tables, "mixed": meta.dec_block_tables}.get(meta.mode)
            if kv_caches:
                meta = copy(meta)
                meta.steady = meta.mode != "decode" and _eight_bits(kv_caches[0])
                if tables is not None:
                    meta.marks = ops.decode_marks(
                        self.spec.n_heads // pdist.tp_world_size(), kv_caches[0][0], tables)
        # layers that somebody watches or has replaced are called and get no parts
        plain = [is_plain(layer, LlamaDecoderLayer) for layer in self.layers] + [True]
        for i, (layer, cache) in enumerate(zip(self.layers, kv_caches)):
            args = x, residual, self.cos_sin, cache, meta
            x, residual = layer.step(*args, plain[i + 1]) if plain[i] else layer(*args)
        x = ops.rmsnorm_residual(x, residual, self.final_norm, self.spec.rms_eps)[0]
        return x  # hidden states [T, H]

    @torch.inference_mode()
    def compute_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        w = self.embed.weight if self.lm_head is None else self.lm_head.weight
        return ops.linear_float(hidden, w)

    @torch.inference_mode()
    def init_random(self, seed: int = 0) -> None:
        """Random-init all weights (synthetic-bench environment: no checkpoints).

        Small params use a CPU generator so CPU and GPU instances of the same
        spec get identical weights (engine equivalence tests); big params
        (>16M elements, e.g. the 8B model's) are generated on-device for
        speed — cross-device bit-equality is irrelevant at that scale.
        """
        gen = torch.Generator(device="cpu").manual_seed(seed)
        dev_gen = None
        for name, p in self.named_parameters():
            if p.dim() >= 2:
                std = p.shape[-1] ** -0.5
                if p.numel() > (1 << 24) and p.device.type != "cpu":
                    if dev_gen is None:
                        dev_gen = torch.Generator(device=p.device).manual_seed(seed)
                    r = torch.randn(p.shape, generator=dev_gen, device=p.device,
                                    dtype=torch.float32)
                else:
                    r = torch.randn(p.shape, generator=gen, dtype=torch.float32)
                p.copy_(r.mul_(std).to(p.dtype))
            else:
                p.copy_(torch.ones(p.shape, dtype=p.dtype))
