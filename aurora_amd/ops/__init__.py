"""Op dispatch layer.

On CUDA (= ROCm/HIP) tensors every op routes to the in-tree gfx950 HIP
extensions ``aurora_amd._hip_ops`` (decoders) and ``aurora_amd._hip_aux``
(encoder, vector search) and FAILS LOUDLY if one is not built —
there is deliberately no silent eager fallback on the GPU path (the whole
point is the CDNA4 kernels; a quiet PyTorch fallback would fake GPU tests).
On CPU tensors ops route to the fp32 reference (``torch_ref``) so the full
pipeline runs and is testable in CPU-only CI.

Build the extensions with ``python setup.py build_ext --inplace`` (hipcc,
``--offload-arch=gfx950``) — see ``aurora_amd/ops/csrc/``.
"""
from __future__ import annotations

from typing import NamedTuple, Optional, Tuple

import torch
import torch.nn.functional as F

from . import torch_ref

_hip = None
_hip_import_error: Optional[BaseException] = None
try:  # the in-tree extensions: aurora_amd/_hip_ops*.so, _hip_aux*.so
    from aurora_amd import _hip_ops as _hip  # type: ignore
except Exception as e:  # pragma: no cover - exercised only when unbuilt
    _hip_import_error = e
_aux = None
_aux_import_error: Optional[BaseException] = None
try:
    from aurora_amd import _hip_aux as _aux  # type: ignore
except Exception as e:  # pragma: no cover - exercised only when unbuilt
    _aux_import_error = e


def hip_available() -> bool:
    return _hip is not None


def _require_hip(op: str, aux: bool = False):
    module, error = (_aux, _aux_import_error) if aux else (_hip, _hip_import_error)
    if module is None:
        raise RuntimeError(
            f"aurora_amd HIP extension is not built but op '{op}' was called on a GPU "
            f"tensor. Build it in-tree with `python setup.py build_ext --inplace` "
            f"(PYTORCH_ROCM_ARCH=gfx950). Import error: {error!r}"
        )
    return module


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-5) -> torch.Tensor:
    if x.is_cuda:
        return _require_hip("rmsnorm").rmsnorm(x.contiguous(), weight, eps)
    return torch_ref.rmsnorm(x, weight, eps)


def rmsnorm_residual(
    x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float = 1e-5
) -> Tuple[torch.Tensor, torch.Tensor]:
    if x.is_cuda:
        m = _require_hip("rmsnorm_residual")
        return m.rmsnorm_residual(x.contiguous(), residual, weight, eps)
    return torch_ref.rmsnorm_residual(x, residual, weight, eps)


def rope_apply(
    q: torch.Tensor, k: torch.Tensor, positions: torch.Tensor, cos_sin: torch.Tensor
) -> Tuple[torch.Tensor, torch.Tensor]:
    if q.is_cuda:
        m = _require_hip("rope_apply")
        q = q.contiguous()
        k = k.contiguous()
        m.rope_apply_(q, k, positions.to(torch.int32), cos_sin)  # in-place
        return q, k
    return torch_ref.rope_apply(q, k, positions, cos_sin)


def rope_apply_(
    q: torch.Tensor, k: torch.Tensor, positions: torch.Tensor, cos_sin: torch.Tensor
) -> None:
    """``rope_apply`` in place, on rows that may be strided (columns of a projection)."""
    if q.is_cuda:
        _require_hip("rope_apply_").rope_apply_(q, k, positions.to(torch.int32), cos_sin)
        return
    for x, y in zip((q, k), torch_ref.rope_apply(q, k, positions, cos_sin)):
        x.copy_(y)


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    if gate_up.is_cuda:
        return _require_hip("silu_mul").silu_mul(gate_up.contiguous())
    return torch_ref.silu_mul(gate_up)


def attention_prefill(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    cu_seqlens: torch.Tensor,
    scale: float,
    causal: bool = True,
) -> torch.Tensor:
    if q.is_cuda:
        m = _require_hip("attention_prefill", aux=True)
        # rows may be strided
        return m.attention_prefill(q, k, v, cu_seqlens.to(torch.int32).contiguous(),
                                   float(scale), bool(causal))
    return torch_ref.attention_prefill(q, k, v, cu_seqlens, scale, causal)


def attention_prefill_turned(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    cos_sin: torch.Tensor,
    cu_seqlens: torch.Tensor,
    scale: float,
    causal: bool = True,
) -> torch.Tensor:
    """``attention_prefill`` of queries and keys that are rotated first, each by its place in
    its sequence; ``cos_sin`` reaches as far as the longest. They stay as they are."""
    if q.is_cuda:
        m = _require_hip("attention_prefill_turned", aux=True)
        return m.attention_prefill_turned(
            q, k, v, cos_sin.to(torch.float32).contiguous(),
            cu_seqlens.to(torch.int32).contiguous(), float(scale), bool(causal))
    begin = torch.repeat_interleave(cu_seqlens[:-1], cu_seqlens.diff())
    q, k = rope_apply(q, k, torch.arange(q.shape[0], device=q.device) - begin, cos_sin)
    return torch_ref.attention_prefill(q, k, v, cu_seqlens, scale, causal)


def attention_prefill_paged(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    cu_seqlens_q: torch.Tensor,
    context_lens: torch.Tensor,
    scale: float,
    out: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """``out``: where the results go, contiguous and shaped as ``q``."""
    if q.is_cuda:
        m = _require_hip("attention_prefill_paged")
        return m.attention_prefill_paged(
            q.contiguous(), k_cache, v_cache, block_tables.to(torch.int32),
            cu_seqlens_q.to(torch.int32), context_lens.to(torch.int32), float(scale), out,
        )
    y = torch_ref.attention_prefill_paged(
        q, k_cache, v_cache, block_tables, cu_seqlens_q, context_lens, scale
    )
    return y if out is None else out.copy_(y)


def kv_cache_write(
    k: torch.Tensor, v: torch.Tensor,
    k_cache: torch.Tensor, v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> None:
    if k.is_cuda:
        m = _require_hip("kv_cache_write")
        m.kv_cache_write(k.contiguous(), v.contiguous(), k_cache, v_cache,
                         slot_mapping.to(torch.int32))
        return
    torch_ref.kv_cache_write(k, v, k_cache, v_cache, slot_mapping)


def paged_attention_decode(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    context_lens: torch.Tensor,
    scale: float,
    out: Optional[torch.Tensor] = None,
    marks: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """``out``: where the results go, contiguous and shaped as ``q``; ``marks``: of
    ``decode_marks`` for this batch."""
    if q.is_cuda:
        m = _require_hip("paged_attention_decode")
        return m.paged_attention_decode(
            q.contiguous(), k_cache, v_cache,
            block_tables.to(torch.int32), context_lens.to(torch.int32), float(scale), out,
            marks,
        )
    y = torch_ref.paged_attention_decode(q, k_cache, v_cache, block_tables, context_lens, scale)
    return y if out is None else out.copy_(y)


def decode_marks(heads: int, k_cache: torch.Tensor, block_tables: torch.Tensor,
                 window: int = 0, chunk: int = 0) -> Optional[torch.Tensor]:
    """Zeros by which decode attention finds out that all stretches of a context are done.
    It leaves zeros behind, so the layers of a step, which follow each other on one stream,
    share them. None where contexts stay whole."""
    if not k_cache.is_cuda:
        return None
    n = _require_hip("decode_marks").decode_marks(
        block_tables.shape[0], heads, k_cache.shape[1],
        block_tables.shape[1] * k_cache.shape[2], window, chunk)
    return torch.zeros(n, dtype=torch.int32, device=k_cache.device) if n else None


def fused_rope_kv_write(qkv, positions, slots, cos_sin, k_cache, v_cache,
                        n_heads: int, n_kv_heads: int, bias=None):
    """Split fused qkv output, RoPE q/k, scatter k/v into the paged cache;
    returns contiguous roped q [T, Hq, D].  One kernel on GPU; composed
    reference ops on CPU. ``qkv`` may be a product in parts (``linear_parts``);
    ``bias`` is added to it first."""
    if qkv.is_cuda:
        m = _require_hip("fused_rope_kv_write")
        return m.fused_rope_kv_write(qkv.contiguous(), positions.to(torch.int32),
                                     slots.to(torch.int32), cos_sin,
                                     k_cache, v_cache, n_heads, n_kv_heads, bias)
    if bias is not None:
        qkv = qkv + bias
    T = qkv.shape[0]
    D = k_cache.shape[3]
    q = qkv[:, : n_heads * D].reshape(T, n_heads, D)
    k = qkv[:, n_heads * D: (n_heads + n_kv_heads) * D].reshape(T, n_kv_heads, D)
    v = qkv[:, (n_heads + n_kv_heads) * D:].reshape(T, n_kv_heads, D)
    q, k = torch_ref.rope_apply(q, k, positions, cos_sin)
    torch_ref.kv_cache_write(k, v, k_cache, v_cache, slots)
    return q


def fresh_attention_decode(qkv, bias, positions, slots, cos_sin, k_cache, v_cache, block_tables,
                           context_lens, n_heads: int, scale: float, marks=None) -> torch.Tensor:
    """``fused_rope_kv_write`` and ``paged_attention_decode`` of rows that are the last tokens of
    different sequences, each at the place and position that its table and context say; in one
    kernel where it has a form."""
    n_kv_heads = k_cache.shape[1]
    if qkv.is_cuda:
        m = _require_hip("fresh_attention_decode")
        out = m.fresh_attention_decode(qkv, bias, cos_sin, k_cache, v_cache, block_tables,
                                       context_lens, n_heads, float(scale), marks)
        if out is not None:
            return out
    q = fused_rope_kv_write(qkv, positions, slots, cos_sin, k_cache, v_cache, n_heads,
                            n_kv_heads, bias)
    return paged_attention_decode(q, k_cache, v_cache, block_tables, context_lens, scale,
                                  marks=marks)


def embed_pool(hidden: torch.Tensor, cu_seqlens: torch.Tensor) -> torch.Tensor:
    if hidden.is_cuda:
        return _require_hip("embed_pool", aux=True).embed_pool(hidden.contiguous(), cu_seqlens.to(torch.int32))
    return torch_ref.embed_pool(hidden, cu_seqlens)


def knn_topk(query: torch.Tensor, docs: torch.Tensor, k: int):
    if query.is_cuda:
        return _require_hip("knn_topk", aux=True).knn_topk(query.contiguous(), docs, int(k))
    return torch_ref.knn_topk(query, docs, k)


def linear(x: torch.Tensor, weight: torch.Tensor, steady: bool = False) -> torch.Tensor:
    """Bias-free linear: own kernels on the GPU where they win (``own_product``),
    hipBLASLt otherwise. ``steady``: the sums keep their order, for what an 8-bit cache is
    filled with, whose bytes show it."""
    y = _hip.own_product(x, weight, 4 if steady else 0) if x.is_cuda and _hip is not None else None
    return F.linear(x, weight) if y is None else y


def linear_float(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``linear(x, weight).float()``, rounded all the same; without a pass of its own where few
    rows have many outputs."""
    y = _hip.own_product(x, weight, 3) if x.is_cuda and _hip is not None else None
    return linear(x, weight).float() if y is None else y


class Unnormed(NamedTuple):
    """A row whose norm is done by the product that reads it (``norm_ahead``)."""

    parts: torch.Tensor
    residual: torch.Tensor
    weight: torch.Tensor
    eps: float
    sum: torch.Tensor  # the new residual, written by that product

    @property
    def shape(self):
        return self.residual.shape


def norm_ahead(x, residual, weight, eps, reader: Optional[torch.Tensor], silu: bool,
               steady: bool = False):
    """``rmsnorm_residual`` for ``linear_parts``, or with ``silu`` ``linear_silu_mul``, by
    ``reader``, the only reader of the rows: a single row in parts is left to it. ``steady``
    as the product is told."""
    if (reader is not None and x.is_cuda and x.dim() == 3 and x.shape[1] == 1
            and _require_hip("norm_ahead").norms_row(x, residual, weight, reader, silu, steady)):
        new = torch.empty_like(residual)
        return Unnormed(x, residual, weight, float(eps), new), new
    return rmsnorm_residual(x, residual, weight, eps)


def linear_parts(x, weight: torch.Tensor, steady: bool = False) -> torch.Tensor:
    """As ``linear``, but where the product of few rows is cut along K its parts
    [S, T, N] in float32, for a reader that adds and rounds them itself
    (``rmsnorm_residual``, ``fused_rope_kv_write``). ``x``: rows, or one of
    ``norm_ahead``."""
    if isinstance(x, Unnormed):
        return _hip.one_row_product(*x, weight, False, steady)
    y = _hip.own_product(x, weight, 5 if steady else 1) if x.is_cuda and _hip is not None else None
    return F.linear(x, weight) if y is None else y


def linear_norm_parts(x, weight: torch.Tensor, beside_experts: bool = False) -> torch.Tensor:
    """``linear_parts`` for ``residual_rmsnorm``, which adds parts up itself where its threads
    hold a row: more than 256 rows up to 2048 wide, ``beside_experts``' rows up to 4096."""
    held = x.shape[0] <= 256 or weight.shape[0] <= (4096 if beside_experts else 2048)
    return (linear_parts if held else linear)(x, weight)


def linear_silu_mul(x, weight: torch.Tensor, steady: bool = False) -> torch.Tensor:
    """silu(gate) * up of the products with gate's rows, then up's; in one kernel where that
    is faster. ``x``: rows, or one of ``norm_ahead``."""
    if isinstance(x, Unnormed):
        return _hip.one_row_product(*x, weight, True)
    y = _hip.own_product(x, weight, 2) if x.is_cuda and _hip is not None else None
    return silu_mul(linear(x, weight, steady)) if y is None else y


def has_moe_grouped(x: torch.Tensor, router: Optional[torch.Tensor] = None) -> bool:
    """True when the grouped expert kernels serve this tensor, with ``router`` the router
    kernel too: 512 experts at most, weights of the tensor's type. Eight experts of 4096 x
    14336, two each: 32 rows 833 -> 516 us against products packed for decoding, 300 rows
    1600 -> 730 and 8192 rows 6210 -> 5740 us against a library product per expert."""
    import os
    return (x.is_cuda and x.dtype == torch.bfloat16 and _hip is not None
            and x.shape[1] % 64 == 0 and not (x.is_contiguous() and x.data_ptr() % 16)
            and (router is None or (router.shape[0] <= 512 and router.dtype == x.dtype
                                    and router.is_contiguous()))
            and os.environ.get("AURORA_MOE_GROUPED", "1") != "0")


def moe_silu_glu(x: torch.Tensor, router: torch.Tensor, top: int, w_gate_up: torch.Tensor,
                 w_down: torch.Tensor) -> torch.Tensor:
    """Top-k routed silu GLU experts of bf16 GPU rows: fp32 router and softmax over the
    chosen, rows sorted by expert on the device, two grouped products, weighted fp32 sum.
    Nothing is read back and all shapes are static."""
    m = _require_hip("moe_silu_glu")
    x = x.contiguous()
    sel, weights = m.moe_route(x, router, None, top)
    y, place = m.moe_silu_glu(x, sel, w_gate_up, w_down)
    return m.moe_combine(y, place, weights)


def moe_grouped_gemm(xp: torch.Tensor, w: torch.Tensor, starts: torch.Tensor,
                     counts: torch.Tensor) -> torch.Tensor:
    """Packed per-expert GEMM: yp[A, N] with tokens sorted by expert.
    Requires per-expert counts <= 256 (the decode regime; prefill uses
    per-expert dense GEMMs)."""
    return _require_hip("moe_grouped_gemm").moe_grouped_gemm(
        xp.contiguous(), w, starts, counts)


def pack_batch(ids, first, end, pages, states, prompts: int, page: int, device):
    """A step's ids, positions, cache slots and tables on the GPU, or None where its lists
    hold anything but plain integers (the extension's header has the order)."""
    return _require_hip("pack_batch").pack_batch(ids, first, end, pages, states, prompts, page,
                                                 torch.device(device))


def pack_rows(rows, device):
    """A list of plain integers on the GPU, without waiting for what runs there, or None."""
    return _require_hip("pack_rows").pack_rows(list(rows), torch.device(device))


def stage_decode(seqs, ids, host, keys, inputs, width, page, scratch_page, scratch_slot) -> bool:
    """A captured decode step's inputs from its sequences, or False as ``pack_batch``."""
    return _require_hip("stage_decode").stage_decode(
        list(seqs), ids, host, keys, inputs, width, page, scratch_page, scratch_slot)


def pack_texts(texts, most: int, device):
    """Ids, begins and positions of texts on the GPU, or None as ``pack_batch``."""
    return _require_hip("pack_texts").pack_texts(texts, most, torch.device(device))


def softmax_sample(logits, temperature, top_p, top_k, generator=None):
    # Sampling is [B, V] with B small; keep it in torch on both devices for now
    # (the GPU cost is one softmax over V — negligible next to the forward).
    return torch_ref.softmax_sample(logits, temperature, top_p, top_k, generator)


from .sequence import (  # noqa: E402
    ConvHeadsParams,
    DeltaRuleParams,
    HeadDeltaParams,
    LatentFrontParams,
    LatentParams,
    MatrixMemoryParams,
    NormedHeadsParams,
    RetentionParams,
    Segment,
    bias_kv_write,
    biased_attention,
    cache_head_dims,
    conv_qkv,
    delta_rule,
    embed_pairs,
    gelu,
    head_delta_rule,
    latent_attention,
    latent_front,
    latent_head_width,
    latent_rotary_widths,
    latent_width,
    latent_write,
    matrix_memory,
    moe_clamped_glu,
    moe_grouped_glu,
    moe_softmax_relu2,
    normed_qkv,
    output_norm,
    relu2,
    residual_rmsnorm,
    residual_rmsnorm_conv,
    retention,
    short_conv_add,
    silu_glu,
    xielu,
)
