"""Performance cases: what a user of the framework has it do on one GPU.

Serving: steps of the engine (``LLMEngine.execute``) for dense, routed and layer-listed
decoders, with weights at full width and as many layers as a case says. A step runs the
next tokens of some prompts, one token of every sequence that is decoding, or both, over
the paged cache and the recurrent states. Retrieval: texts to embeddings
(``SentenceEncoder.encode_ids``) and the nearest of many embeddings (``ops.knn_topk``).

Everything is made from a seed on the device. What lies in the caches before a step is
drawn at random, so that long contexts need no prompt of their own to be run first.
Tokens are drawn unevenly, and routed models send a token to experts of its own, as
trained routers do, so the experts' loads are uneven and no choice hangs on a rounding.
"""
import math
import os
import zlib

import torch

from aurora_amd import ops
from aurora_amd.engine.engine import EngineConfig, LLMEngine, Sequence
from aurora_amd.engine.sampling_params import SamplingParams
from aurora_amd.models.config import HybridSpec, ModelSpec, kikalix_layers, senotar_spec
from aurora_amd.models.encoder import SentenceEncoder
from aurora_amd.models.hybrid import HybridForCausalLM
from aurora_amd.models.llama import LlamaForCausalLM

DEV = "cuda"
PAGE = 256
#: a decoding batch starts over from the stored contexts after so many steps
DECODE_CYCLE = 64

#: width, heads, kv heads, head width, ff, vocabulary, rope base, eps, tied, qkv bias, experts
LLAMA = {
    "llama3-8b": (4096, 32, 8, 128, 14336, 128256, 5e5, 1e-5, False, False, 0),
    "llama3.2-1b": (2048, 32, 8, 64, 8192, 128256, 5e5, 1e-5, True, False, 0),
    "qwen2-7b": (3584, 28, 4, 128, 18944, 152064, 1e6, 1e-6, False, True, 0),
    "mixtral-8x7b": (4096, 32, 8, 128, 14336, 32000, 1e6, 1e-5, False, False, 8),
}
#: width, heads, kv heads, experts, top, ff
KIKALIX = {
    "kikalix-4096": (4096, 32, 8, 8, 2, 14336),
    "kikalix-2048": (2048, 16, 8, 64, 6, 1408),
    "kikalix-1024": (1024, 8, 2, 16, 2, 512),
}
#: width, heads, latent rank, ff
SENOTAR = {
    "senotar-4096": (4096, 32, 512, 14336),
    "senotar-2048": (2048, 16, 512, 5632),
    "senotar-1024": (1024, 16, 256, 2816),
}
HYBRID_VOCAB, HYBRID_POSITIONS = 32000, 8192
KIKALIX_PATTERN, SENOTAR_PATTERN = "pppr", "osos"
WINDOW, RANK, TAPS, BUCKETS, LIMIT = 1024, 128, 4, 65521, 7.0


def _step(name, model, layers, prompts=0, tokens=(0, 0), past=(0, 0), decodes=0,
          context=(0, 0), cache="bf16"):
    """A step: ``prompts`` portions of tokens[0]..tokens[1] tokens behind past[0]..past[1]
    cached ones, and ``decodes`` sequences at context[0]..context[1] cached tokens."""
    case = {"kind": "step", "model": model, "layers": layers, "prompts": prompts,
            "tokens_lo": tokens[0], "tokens_hi": tokens[1], "past_lo": past[0],
            "past_hi": past[1], "decodes": decodes, "context_lo": context[0],
            "context_hi": context[1], "cache": cache}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one analyst chatting: the latency of a token of the agent model
        _step("chat token of 1 sequence", "llama3-8b", 16, decodes=1, context=(777, 777)),
        # many investigations at once, a few turns into their contexts
        _step("decode of 96 investigations", "llama3-8b", 16, decodes=96, context=(500, 2900)),
        # the small triage model with the eight-bit cache that doubles its capacity
        _step("decode of 23 triages with fp8 cache", "llama3.2-1b", 16, decodes=23,
              context=(300, 5000), cache="fp8"),
        # first prompts of new investigations, packed into one batch
        _step("8 first prompts", "llama3-8b", 8, prompts=8, tokens=(400, 1100)),
        # one portion of a long log pasted behind an already long context
        _step("one portion behind a long context", "llama3-8b", 4, prompts=1, tokens=(4096, 4096),
              past=(22000, 22000)),
        # tool results of three investigations join a running batch of a routed model
        _step("tool results beside decodes", "mixtral-8x7b", 2, prompts=3, tokens=(350, 650),
              past=(800, 2200), decodes=41, context=(700, 2600)),
        # routed decoding: every expert's weights for a few tokens each
        _step("routed decode of 32 sequences", "mixtral-8x7b", 2, decodes=32,
              context=(600, 2500)),
        # a prompt batch of a layer-listed decoder: window attention, recurrences, experts
        _step("4 prompts recurrent and routed", "kikalix-4096", 4, prompts=4,
              tokens=(1900, 2048)),
        # the same design with many narrow experts, decoding
        _step("recurrent decode of 64 sequences", "kikalix-2048", 4, decodes=64,
              context=(1500, 2500)),
        # latent attention: prompt portions behind a context beside decoding sequences
        _step("latent portions beside decodes", "senotar-4096", 4, prompts=2,
              tokens=(500, 1500), past=(0, 2000), decodes=30, context=(1000, 3000)),
        # a document's chunks on their way into the retrieval index
        {"name": "embed 200 chunks", "kind": "encode", "texts": 200, "lo": 20, "hi": 256},
        # a query against a million embeddings, held as the index holds them
        {"name": "nearest of a million", "kind": "search", "docs": 1_000_000, "queries": 1,
         "k": 20, "dtype": "float32"},
    ]


def _log(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def _span(rng, lo, hi):
    a, b = sorted((_log(rng, lo, hi), _log(rng, lo, hi)))
    return a, b


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "encode", "search"])
    if kind == "encode":
        lo, hi = _span(rng, 4, 256)
        return {"kind": "encode", "texts": _log(rng, 1, 400), "lo": lo, "hi": hi}
    if kind == "search":
        return {"kind": "search", "docs": _log(rng, 5000, 1_000_000),
                "queries": _log(rng, 1, 8), "k": _log(rng, 1, 40),
                "dtype": rng.choice(["float32", "bfloat16"])}
    model = rng.choice([*LLAMA, *LLAMA, *KIKALIX, *SENOTAR])
    layers = 2 if model.startswith("mixtral") else 4
    # sequences of layer-listed models and their caches stay under their positions
    far = 6000 if model not in LLAMA else 12000
    prompts = decodes = 0
    tokens = past = context = (0, 0)
    if kind != "decode":
        prompts = _log(rng, 1, 8)
        tokens = _span(rng, 16, 6000 // prompts)
        # a recurrent state cannot be made up for a portion; its prompts are whole
        if model not in KIKALIX and rng.random() < 0.5:
            past = _span(rng, 64, far // 2 if model not in LLAMA else far)
            tokens = (min(tokens[0], 1500), min(tokens[1], 1500))
    if kind != "prompt":
        decodes = _log(rng, 1, 128 if kind == "decode" else 48)
        context = _span(rng, 30, max(60, min(far, 200_000 // decodes)))
    cache = "fp8" if model in LLAMA and rng.random() < 0.2 else "bf16"
    return _step(None, model, layers, prompts, tokens, past, decodes, context, cache)


# ---- what a case consists of ------------------------------------------------------

def _spread(n, lo, hi):
    """n uneven whole numbers from lo to hi."""
    return [lo + int((hi - lo) * (((i + 1) * 0.6180339887) % 1.0) + 0.5) for i in range(n)]


def _portions(case):
    """(cached tokens, new tokens) of every sequence of a step, prompts first."""
    out = list(zip(_spread(case["prompts"], case["past_lo"], case["past_hi"]),
                   _spread(case["prompts"], case["tokens_lo"], case["tokens_hi"])))
    return out + [(c, 1) for c in _spread(case["decodes"], case["context_lo"],
                                          case["context_hi"])]


def _random(seed, name, shape, scale=1.0):
    """Normal numbers of a name, the same wherever they are asked for."""
    g = torch.Generator(device=DEV).manual_seed(zlib.crc32(f"{name}/{seed}".encode()))
    return torch.randn(shape, generator=g, device=DEV).mul_(scale)


def _tokens(seed, name, n, vocab):
    g = torch.Generator().manual_seed(zlib.crc32(f"{name}/{seed}".encode()))
    return (torch.rand(n, generator=g).pow(2) * (vocab - 1)).long()  # uneven


def _experts(model):
    if model in LLAMA:
        return LLAMA[model][10]
    return KIKALIX[model][3] if model in KIKALIX else 0


def _sizes(model):
    """(width, vocabulary)"""
    if model in LLAMA:
        return LLAMA[model][0], LLAMA[model][5]
    return (KIKALIX if model in KIKALIX else SENOTAR)[model][0], HYBRID_VOCAB


def _weight(case, seed, name, shape):
    """The weight of a name, in the model's own scale. The first columns of a routed
    model's stream hold every token's liking for each expert: routers read them and no
    output projection writes them."""
    experts = _experts(case["model"])
    if "router.b" in name:
        return _random(seed, name, shape, 0.01)
    if "router" in name:
        w = torch.zeros(shape, device=DEV)
        order = _random(seed, name, (experts,)).argsort()
        w[torch.arange(experts, device=DEV), order] = 1.0
        return w
    if name.endswith("norm") or ".norm" in name:
        offset = 0.0 if case["model"] in KIKALIX and not name.endswith("right.norm") else 1.0
        w = _random(seed, name, shape, 0.0 if name.endswith("right.norm") else 0.1) + offset
        if experts and shape[0] == _sizes(case["model"])[0]:
            w[:experts] = offset
        return w
    if len(shape) == 1 or name.endswith(("A_log", "sink")):
        if name.endswith("dt_bias"):
            return _random(seed, name, shape) - 3.0
        return _random(seed, name, shape, {"A_log": 0.5, "sink": 1.0, "act": 0.5}.get(
            name.rsplit(".", 1)[-1], 0.1))
    w = _random(seed, name, shape, shape[-1] ** -0.5)
    if name.startswith(("embed", "bigram")):
        w = w * shape[-1] ** 0.5
        if experts:
            rung = torch.special.ndtri((torch.arange(experts, device=DEV) + 0.5) / experts)
            w[:, :experts] = rung[_random(seed, name + ".liking", (shape[0], experts))
                                  .argsort(-1)]
    elif name.endswith("canon1"):
        w = w * (0.3 * shape[-1] ** 0.5)
    elif experts and name.endswith((".o", ".down", "o_proj.weight", "down.weight")):
        w[:experts] = 0.0
    return w


# ---- models -----------------------------------------------------------------------

def _llama_spec(case):
    w, h, kv, d, ff, vocab, base, eps, tied, bias, experts = LLAMA[case["model"]]
    return ModelSpec(name=case["model"], hidden_size=w, n_layers=case["layers"], n_heads=h,
                     n_kv_heads=kv, head_dim=d, intermediate_size=ff, vocab_size=vocab,
                     rope_theta=base, rms_eps=eps, max_position=32768, tie_embeddings=tied,
                     qkv_bias=bias, n_experts=experts)


def _hybrid_spec(case):
    n = case["layers"]
    if case["model"] in SENOTAR:
        w, h, rank, ff = SENOTAR[case["model"]]
        return senotar_spec(case["model"], (SENOTAR_PATTERN * n)[:n], width=w,
                            vocab=HYBRID_VOCAB, heads=h, dim=w // h, vdim=w // h,
                            kv_rank=rank, ff=ff, taps=TAPS, buckets=BUCKETS,
                            max_position=HYBRID_POSITIONS)
    w, h, kv, experts, top, ff = KIKALIX[case["model"]]
    d = w // h
    return HybridSpec(
        name=case["model"], hidden_size=w, vocab_size=HYBRID_VOCAB,
        max_position=HYBRID_POSITIONS, layers=kikalix_layers(
            (KIKALIX_PATTERN * n)[:n], heads=h, kv_heads=kv, dim=d, vdim=d, window=WINDOW,
            d_heads=h // 2, d_kv_heads=h // 2, d_dim=d, d_vdim=d, rank=RANK, r_heads=h // 2,
            r_dim=d, r_vdim=2 * d, experts=experts, top=top, ff=ff, conv=TAPS, limit=LIMIT))


@torch.inference_mode()
def _model(case, seed):
    with torch.device(DEV):  # nothing is initialised twice or on the host
        if case["model"] in LLAMA:
            model = LlamaForCausalLM(_llama_spec(case), dtype=torch.bfloat16)
        else:
            model = HybridForCausalLM(_hybrid_spec(case), dtype=torch.bfloat16, device=DEV)
    if case["model"] in LLAMA:
        for name, p in model.named_parameters():
            p.copy_(_weight(case, seed, name, tuple(p.shape)))
    else:
        shapes = {n: tuple(t.shape) for n, t in model.named_tensors().items()}
        model.load_tensors(lambda n: _weight(case, seed, n, shapes[n]))
    return model.eval()


def _cached(case, seed, layer, part, rows, shape):
    """What the cache holds of ``rows`` tokens before the step, in its own type."""
    x = _random(seed, f"cache{layer}{part}", (rows, *shape))
    return x.to(torch.float8_e4m3fn if case["cache"] == "fp8" else torch.bfloat16)


def _state_scale(entry):
    return 0.1 if entry.dim() == 4 else 1.0  # matrices; last inputs


def prepare(case, seed):
    return {"encode": _prepare_encode, "search": _prepare_search,
            "step": _prepare_step}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


@torch.inference_mode()
def _prepare_step(case, seed):
    model = _model(case, seed)
    portions, n = _portions(case), case["prompts"]
    room = [past + new + (DECODE_CYCLE if i >= n else 0) + 1
            for i, (past, new) in enumerate(portions)]
    pages = [-(-r // PAGE) for r in room]
    before = os.environ.get("AURORA_KV_FP8")
    os.environ["AURORA_KV_FP8"] = "1" if case["cache"] == "fp8" else "0"
    try:
        engine = LLMEngine(EngineConfig(
            model=case["model"], page_size=PAGE, kv_cache_pages=sum(pages) + 1,
            max_num_seqs=len(portions), state_slots=len(portions),
            max_model_len=max(4096, max(pages) * PAGE), prefix_cache=False), model=model)
    finally:
        if before is None:
            del os.environ["AURORA_KV_FP8"]
        else:
            os.environ["AURORA_KV_FP8"] = before
    # rows of a captured batch that no sequence fills decode token 0, not what an engine of
    # another vocabulary may have left in the pinned memory
    engine._host_i64.zero_()
    vocab, seqs, nexts = _sizes(case["model"])[1], [], []
    for i, ((past, new), p) in enumerate(zip(portions, pages)):
        ids = _tokens(seed, f"ids{i}", past + max(new, DECODE_CYCLE), vocab).tolist()
        s = Sequence(f"s{i}", ids[:past + (new if i < n else 0)], SamplingParams())
        s.pages, s.num_cached = engine.kv.alloc(p), past
        if engine.states:
            s.state_slot = engine.states.alloc()
        seqs.append(s)
        nexts.append(ids[past:past + DECODE_CYCLE])
    place = torch.tensor([(s.pages[t // PAGE], t % PAGE) for s, (past, _) in
                          zip(seqs, portions) for t in range(past)],
                         dtype=torch.long, device=DEV).view(-1, 2)
    for layer, caches in enumerate(engine.kv.caches):
        for part, cache in zip("kv", caches):
            raw = cache.view(torch.uint8) if case["cache"] == "fp8" else cache
            if cache.shape[3]:
                rows = _cached(case, seed, layer, part, len(place),
                               (cache.shape[1], cache.shape[3]))
                raw[place[:, 0], :, place[:, 1]] = rows.view(raw.dtype)
    for i, entries in enumerate(engine.states.states):
        for j, t in enumerate(entries):
            if t.dtype == torch.int32:  # a pair embedding's last tokens
                for s, (past, _) in zip(seqs, portions):
                    t[s.state_slot] = s.token_ids[past - 1] if past else 0
                continue
            fill = _random(seed, f"state{i}.{j}", (len(seqs), *t.shape[1:]), _state_scale(t))
            t[[s.state_slot for s in seqs]] = fill.to(t.dtype)
    ends, end = [], 0
    for _, new in portions:
        end += new
        ends.append(end - 1)
    caches = [t.view(torch.uint8) if case["cache"] == "fp8" else t
              for pair in engine.kv.caches for t in pair if t.numel()]
    states = [t for entries in engine.states.states for t in entries]
    return {"run": _run_step, "engine": engine, "prompts": seqs[:n], "decodes": seqs[n:],
            "past": [p for p, _ in portions], "nexts": nexts[n:], "rows": ends, "at": 0,
            "chunks": [new for _, new in portions[:n]], "caches": caches, "states": states}


def _run_step(state):
    prompts, n = state["prompts"], len(state["prompts"])
    for s, past in zip(prompts, state["past"]):
        s.num_cached = past
    if state["decodes"]:
        if state["at"] == DECODE_CYCLE:  # a new batch over the same contexts
            again = []
            for s, past in zip(state["decodes"], state["past"][n:]):
                t = Sequence(s.req_id, s.token_ids[:past], s.params)
                t.pages, t.num_cached, t.state_slot = s.pages, past, s.state_slot
                again.append(t)
            state["decodes"], state["at"] = again, 0
        for s, ids in zip(state["decodes"], state["nexts"]):
            s.token_ids.append(ids[state["at"]])
        state["at"] += 1
    logits = state["engine"].execute(prompts, state["chunks"], state["decodes"],
                                     state["rows"])
    return {"logits": logits, "caches": state["caches"], "states": state["states"]}


def _texts(case, seed):
    return [_tokens(seed, f"text{i}", n, 30000).tolist()
            for i, n in enumerate(_spread(case["texts"], case["lo"], case["hi"]))]


@torch.inference_mode()
def _prepare_encode(case, seed):
    with torch.device(DEV):
        encoder = SentenceEncoder("bge-base", dtype=torch.bfloat16, device=DEV)
    for name, p in encoder.named_parameters():
        p.copy_(_weight({"model": "senotar-1024"}, seed, name, tuple(p.shape)))
    return {"run": lambda s: s["encoder"].encode_ids(s["texts"]), "encoder": encoder,
            "texts": _texts(case, seed)}


def _embeddings(case, seed):
    """(queries, documents): unit vectors; every query has a few relatives, the next
    always clearly less alike than the one before."""
    dtype, n, q = getattr(torch, case["dtype"]), case["docs"], case["queries"]

    def unit(x):
        return x / x.norm(dim=-1, keepdim=True)

    docs = unit(_random(seed, "docs", (n, 768)))
    queries = unit(_random(seed, "queries", (q, 768)))
    rank = torch.arange(case["k"] + 8, device=DEV)
    like = (0.95 - 0.015 * rank)[:, None]
    at = _random(seed, "places", (n,)).argsort()[:q * len(rank)].view(q, len(rank))
    for i in range(q):
        d = docs[at[i]]
        side = unit(d - (d @ queries[i])[:, None] * queries[i])
        docs[at[i]] = like * queries[i] + (1 - like * like).sqrt() * side
    return queries.to(dtype), docs.to(dtype)


@torch.inference_mode()
def _prepare_search(case, seed):
    queries, docs = _embeddings(case, seed)
    return {"run": lambda s: dict(zip(("values", "indices"), ops.knn_topk(
        s["queries"], s["docs"], s["k"]))), "queries": queries, "docs": docs, "k": case["k"]}


# ---- what a pass cannot do without --------------------------------------------------

def work(case):
    if case["kind"] == "search":
        size = 768 * (4 if case["dtype"] == "float32" else 2)
        return {"bytes": (case["docs"] + case["queries"]) * size + 16 * case["queries"] * case["k"],
                "flops": 2 * 768 * case["docs"] * case["queries"]}
    if case["kind"] == "encode":
        lens = _spread(case["texts"], case["lo"], case["hi"])
        matrices = 12 * (4 * 768 * 768 + 3 * 768 * 3072)
        return {"bytes": 2 * (matrices + 768 * (sum(lens) + len(lens))),
                "flops": 2 * matrices * sum(lens) + 12 * sum(4 * n * n * 768 for n in lens)}
    portions, model = _portions(case), case["model"]
    tokens = sum(new for _, new in portions)
    width, vocab = _sizes(model)
    flops = 2 * width * vocab * len(portions)
    size = 2 * (vocab * width + tokens * width) + 4 * vocab * len(portions)
    for i in range(case["layers"]):
        f, b = _layer_work(case, i, portions, tokens)
        flops, size = flops + f, size + b
    return {"bytes": size, "flops": flops}


def _seen(portions, window=0):
    """(pairs of a query and a key it sees, keys that some query sees)"""
    pairs = keys = 0
    for past, new in portions:
        for first, count in ((past + 1, new),):
            last = first + count - 1
            if not window or last <= window:
                pairs += (first + last) * count // 2
            else:
                low = max(0, min(count, window - first + 1))
                pairs += (2 * first + low - 1) * low // 2 + (count - low) * window
        keys += min(past + new, window + new) if window else past + new
    return pairs, keys


def _layer_work(case, i, portions, tokens):
    model = case["model"]
    bytes_per = 1 if case["cache"] == "fp8" else 2
    if model in LLAMA:
        w, h, kv, d, ff, _, _, _, _, _, experts = LLAMA[model]
        pairs, keys = _seen(portions)
        matrix, used = w * d * (2 * h + 2 * kv), 1
        if experts:
            used = min(experts, 2 * tokens)
        flops = 2 * tokens * (matrix + 3 * w * ff * (2 if experts else 1)) + 4 * h * d * pairs
        return flops, 2 * (matrix + 3 * w * ff * used) + (keys + tokens) * 2 * kv * d * bytes_per
    if model in SENOTAR:
        w, h, rank, ff = SENOTAR[model]
        own = (SENOTAR_PATTERN * case["layers"])[i] == "o"
        pairs, keys = _seen(portions)
        matrix = 4 * w * w + 2 * w * ff + (w * rank if own else 0) + w * h
        # a head's product over a pair, in its own width; once per token into latents
        flops = 2 * tokens * (matrix + 2 * w * rank) + 4 * w * pairs
        return flops, 2 * (matrix + 2 * w * rank) + 2 * rank * (keys + tokens * own)
    w, h, kv, experts, top, ff = KIKALIX[model]
    used = min(experts, top * tokens)
    flops = 6 * tokens * top * w * ff
    size = 2 * 3 * w * ff * used
    d, sequences = w // h, len(portions)
    fresh = case["prompts"]  # states that are not read
    if (KIKALIX_PATTERN * case["layers"])[i] == "p":
        pairs, keys = _seen(portions, WINDOW)
        half = w // 2
        matrix = w * (w + 2 * kv * d + 3 * half + h // 2 + 2 * RANK + w + half) + RANK * w
        state = 4 * half * d
        flops += 2 * tokens * matrix + 4 * w * pairs + 6 * tokens * half * d
        size += 2 * matrix + (keys + tokens) * 4 * kv * d
    else:
        matrix, state = w * (3 * w + w), 4 * w * d
        flops += 2 * tokens * matrix + 4 * tokens * w * d
        size += 2 * matrix
    return flops, size + state * (2 * sequences - fresh)


def tolerance(case):
    if case["kind"] == "search":  # scores of 32-bit or of 16-bit sums
        return {"rel": 1e-5 if case["dtype"] == "float32" else 1e-2}
    if case["kind"] == "encode":
        return {"rel": 3e-2, "max": 0.3}
    # bf16 activations add their roundings layer by layer (0.0045 * sqrt(layers) off exact
    # were seen); of an 8-bit cache's bytes only the new rows' may round the other way
    rel = 0.015 * case["layers"] ** 0.5
    return {"rel": rel, "max": 10 * rel, "differ": 1e-3}


# ---- the same in 64 bits ------------------------------------------------------------

@torch.inference_mode()
def exact(case, seed):
    if case["kind"] == "search":
        queries, docs = _embeddings(case, seed)
        scores = torch.cat([queries.double() @ d.double().t() for d in docs.split(100_000)], 1)
        return dict(zip(("values", "indices"), scores.topk(min(case["k"], case["docs"]))))
    if case["kind"] == "encode":
        return _exact_encode(case, seed)
    ids = []
    vocab = _sizes(case["model"])[1]
    for i, (past, new) in enumerate(_portions(case)):
        t = _tokens(seed, f"ids{i}", past + max(new, DECODE_CYCLE), vocab)
        ids.append(t[:past + new].to(DEV))
    logits = (_exact_llama if case["model"] in LLAMA else _exact_senotar
              if case["model"] in SENOTAR else _exact_kikalix)(case, seed, ids)
    return {"logits": logits, "caches": None, "states": None}


def _w(case, seed, name, *shape, dtype=torch.bfloat16):
    return _weight(case, seed, name, shape).to(dtype).double()


def _rms(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _rotate(x, positions, dims, base):
    """Halves of the first ``dims`` dimensions of x [n, heads, d] turn together."""
    half = dims // 2
    f = base ** (-torch.arange(half, device=DEV, dtype=torch.float64) * 2 / dims)
    a = positions.double()[:, None, None] * f
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., dims:]], -1)


def _attend(q, k, v, past, scale, slopes=None, window=0, sink=None):
    """q [n, H, d] at positions past.., k and v [past + n, G, *] -> [n, H, e]"""
    n, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = []
    i = torch.arange(past, past + n, device=DEV)[:, None]
    dist = i - torch.arange(past + n, device=DEV)[None, :]
    hidden = (dist < 0) | (dist >= window) if window else dist < 0
    for h in range(H):
        s = (q[:, h] @ k[:, h * G // H].t()) * scale
        if slopes is not None:
            s -= slopes[h] * dist
        s.masked_fill_(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(n, 1)], 1)
        s = torch.softmax(s, -1)
        out.append(s[:, :past + n] @ v[:, h * G // H])
    return torch.stack(out, 1)


def _split(x, ids):
    return x.split([len(i) for i in ids])


def _new(case, ids):
    return [t[past:] for t, (past, _) in zip(ids, _portions(case))]


def _contexts(case, seed, layer, part, shape):
    """Every sequence's cached rows in 64 bits."""
    lens = [past for past, _ in _portions(case)]
    return _cached(case, seed, layer, part, sum(lens), shape).double().split(lens)


def _stored(case, x):
    """New rows as the cache's type holds them."""
    return x.to(torch.float8_e4m3fn).double() if case["cache"] == "fp8" else x


def _last(x, ids):
    return torch.stack([s[-1] for s in _split(x, ids)])


def _routed(x, sel, weight, gate_up, down, experts, act):
    """Sum of the chosen experts' results; their weights are made one expert at a time."""
    out = torch.zeros_like(x)
    for e in range(experts):
        row, place = (sel == e).nonzero(as_tuple=True)
        if len(row):
            g, u = (x[row] @ gate_up(e).t()).chunk(2, -1)
            out.index_add_(0, row, (act(g, u) @ down(e).t()) * weight[row, place, None])
    return out


def _exact_llama(case, seed, ids):
    w, H, G, d, ff, vocab, base, eps, tied, bias, experts = LLAMA[case["model"]]
    silu = torch.nn.functional.silu
    new = _new(case, ids)
    x = _weight(case, seed, "embed.weight", (vocab, w)).bfloat16()[torch.cat(new)].double()
    for i in range(case["layers"]):
        pre = f"layers.{i}."

        def mat(name, *shape):
            return _w(case, seed, pre + name, *shape)

        h = _rms(x, eps) * mat("input_norm", w)
        qkv = h @ mat("attn.qkv_proj.weight", (H + 2 * G) * d, w).t()
        if bias:
            qkv = qkv + mat("attn.qkv_proj.bias", (H + 2 * G) * d)
        ks, vs = (_contexts(case, seed, i, p, (G, d)) for p in "kv")
        outs = []
        for r, (past, n), k0, v0 in zip(_split(qkv, new), _portions(case), ks, vs):
            q, k, v = r.view(n, -1, d).split([H, G, G], 1)
            at = torch.arange(past, past + n, device=DEV)
            q, k = _rotate(q, at, d, base), _rotate(k, at, d, base)
            outs.append(_attend(q, torch.cat([k0, _stored(case, k)]),
                                torch.cat([v0, _stored(case, v)]), past, d ** -0.5))
        x = x + torch.cat(outs).flatten(1) @ mat("attn.o_proj.weight", w, H * d).t()
        h = _rms(x, eps) * mat("post_attn_norm", w)
        if not experts:
            g, u = (h @ mat("mlp.gate_up.weight", 2 * ff, w).t()).chunk(2, -1)
            x = x + (silu(g) * u) @ mat("mlp.down.weight", w, ff).t()
            continue
        top, sel = (h @ mat("mlp.router.weight", experts, w).t()).topk(2, -1)
        x = x + _routed(h, sel, top.softmax(-1),
                        lambda e: mat(f"mlp.experts.{e}.gate_up.weight", 2 * ff, w),
                        lambda e: mat(f"mlp.experts.{e}.down.weight", w, ff), experts,
                        lambda g, u: silu(g) * u)
    x = _rms(_last(x, new), eps) * _w(case, seed, "final_norm", w)
    return x @ _w(case, seed, "embed.weight" if tied else "lm_head.weight", vocab, w).t()


def _conv(x, past, weight):
    """Causal convolution of x [n, C] behind the taps - 1 rows of past; weight [C, taps]"""
    n, taps = x.shape[0], weight.shape[1]
    full = torch.cat([past, x])
    return sum(full[j:j + n] * weight[:, j] for j in range(taps))


def _ring_past(ring, start, taps):
    """The last taps - 1 rows before ``start`` of a ring by position."""
    rows = [ring[(start - j) % len(ring)] if start >= j else torch.zeros_like(ring[0])
            for j in range(taps - 1, 0, -1)]
    return torch.stack(rows).double()


def _exact_kikalix(case, seed, ids):
    w, H, G, experts, top, ff = KIKALIX[case["model"]]
    d, eps, new, portions = w // H, 1e-5, _new(case, ids), _portions(case)
    D, f32, n_seq, longest = H // 2, torch.float32, len(new), max(len(t) for t in new)
    slopes = [2.0 ** (-8.0 * (h + 1) / H) for h in range(H)]
    decay = torch.tensor([1.0 - 2.0 ** (-5 - 3.0 * h / max(D - 1, 1)) for h in range(D)],
                         device=DEV, dtype=torch.float64)
    x = _weight(case, seed, "embed", (HYBRID_VOCAB, w)).bfloat16()[torch.cat(new)].double()

    def batched(parts):  # one padded row of time steps per sequence
        out = torch.zeros(n_seq, longest, *parts[0].shape[1:], device=DEV, dtype=torch.float64)
        for s, p in enumerate(parts):
            out[s, :len(p)] = p
        return out

    def packed(y):
        return torch.cat([y[s, :len(t)] for s, t in enumerate(new)])

    def state(layer, shape):
        S = _random(seed, f"state{layer}.0", (n_seq, *shape), 0.1).double()
        for s, (past, _) in enumerate(portions):
            if past == 0:
                S[s] = 0.0
        return S

    for i in range(case["layers"]):
        pre = f"l{i}.mix."

        def mat(name, *shape, dtype=torch.bfloat16):
            return _w(case, seed, pre + name, *shape, dtype=dtype)

        h = _rms(x, eps) * (1.0 + _w(case, seed, f"l{i}.norm1", w, dtype=f32))
        if (KIKALIX_PATTERN * case["layers"])[i] == "p":
            q, k, v = (h @ mat(f"left.{c}", g * d, w).t() + mat(f"left.{c}.b", g * d, dtype=f32)
                       for c, g in (("q", H), ("k", G), ("v", G)))
            at = sum(p == "p" for p in (KIKALIX_PATTERN * case["layers"])[:i])
            ks, vs = (_contexts(case, seed, at, c, (G, d)) for c in "kv")
            left = torch.cat([
                _attend(a.view(-1, H, d), torch.cat([k0, b.view(-1, G, d)]),
                        torch.cat([v0, c.view(-1, G, d)]), past, d ** -0.5, slopes, WINDOW)
                for a, b, c, k0, v0, (past, _) in zip(
                    _split(q, new), _split(k, new), _split(v, new), ks, vs, portions)])
            left = left.flatten(1) @ mat("left.o", w, H * d).t()
            raw = torch.cat([h @ mat(f"right.{c}", D * d, w).t() for c in "qkv"], 1)
            weight = torch.cat([mat(f"right.{c}.conv", D * d, TAPS, dtype=f32) for c in "qkv"])
            rings = _random(seed, f"state{i}.1", (n_seq, TAPS, 3 * D * d)).bfloat16()
            y = torch.cat([_conv(r, _ring_past(ring, past, TAPS), weight) for r, ring, (past, _)
                           in zip(_split(raw, new), rings, portions)])
            q, k, v = torch.nn.functional.silu(y).view(-1, 3, D, d).unbind(1)
            q, k = (t * torch.rsqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
            beta = torch.sigmoid(h @ mat("right.b", D, w).t())
            u = h @ mat("right.a1", RANK, w).t() @ mat("right.a2", D * d, RANK).t()
            u = torch.nn.functional.softplus(u + mat("right.dt_bias", D * d, dtype=f32))
            g = torch.exp(-mat("right.A_log", D, dtype=f32).exp()[:, None] * u.view(-1, D, d))
            q, k, v, g, beta = (batched(_split(t, new)) for t in (q * d ** -0.5, k, v, g, beta))
            S, out = state(i, (D, d, d)), torch.zeros_like(v)
            for t in range(longest):
                S = S * g[:, t, :, :, None]
                r = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S)[:, :, 0])
                S = S + k[:, t, :, :, None] * r[:, :, None]
                out[:, t] = (q[:, t, :, None] @ S)[:, :, 0]
            gate = torch.sigmoid(h @ mat("right.g1", RANK, w).t() @ mat("right.g2", D * d, RANK).t())
            right = _rms(packed(out), eps) * mat("right.norm", d, dtype=f32)
            right = (right.flatten(1) * gate) @ mat("right.o", w, D * d).t()
            x = x + 0.5 * left + 0.5 * right
        else:
            q, k = (h @ mat(c, D * d, w).t() for c in "qk")
            v, gate = (h @ mat(c, 2 * D * d, w).t() for c in "vg")
            pos = torch.cat([torch.arange(past, past + n, device=DEV) for past, n in portions])
            q, k = (_rotate(t.view(-1, D, d), pos, d, 1e4) for t in (q, k))
            q, k, v = (batched(_split(t, new)) for t in (q, k * d ** -0.5, v.view(-1, D, 2 * d)))
            S, out = state(i, (D, d, 2 * d)), torch.zeros_like(v)
            for t in range(longest):
                S = S * decay[:, None, None] + k[:, t, :, :, None] * v[:, t, :, None]
                out[:, t] = (q[:, t, :, None] @ S)[:, :, 0]
            out = _rms(packed(out), eps).flatten(1) * torch.nn.functional.silu(gate)
            x = x + out @ mat("o", w, 2 * D * d).t()
        pre = f"l{i}.mlp."
        h = _rms(x, eps) * (1.0 + _w(case, seed, f"l{i}.norm2", w, dtype=f32))
        z, sel = (h @ mat("router", experts, w).t() + mat("router.b", experts, dtype=f32)).topk(
            top, -1)
        x = x + _routed(
            h, sel, z.softmax(-1),
            lambda e: torch.cat([mat(f"e{e}.gate", ff, w), mat(f"e{e}.up", ff, w)]),
            lambda e: mat(f"e{e}.down", w, ff), experts,
            lambda g, u: g.clamp(max=LIMIT) * torch.sigmoid(1.702 * g.clamp(max=LIMIT))
            * (u.clamp(-LIMIT, LIMIT) + 1.0))
    x = _rms(_last(x, new), eps) * (1.0 + _w(case, seed, "final.norm", w, dtype=f32))
    return x @ _w(case, seed, "head", HYBRID_VOCAB, w).t()


def _exact_senotar(case, seed, ids):
    w, H, rank, ff = SENOTAR[case["model"]]
    d, eps, new, portions, f32 = w // H, 1e-5, _new(case, ids), _portions(case), torch.float32
    pattern = (SENOTAR_PATTERN * case["layers"])[:case["layers"]]
    table = _weight(case, seed, "embed", (HYBRID_VOCAB, w)).bfloat16()
    pairs = _weight(case, seed, "bigram", (BUCKETS + 1, w)).bfloat16()
    rows = []
    for t, (past, n) in zip(ids, portions):
        row = (torch.cat([t[:1], t[:-1]]) * 31 + t * 17) % BUCKETS
        row[0] = BUCKETS  # nothing before the first
        rows.append(row[past:])
    x = table[torch.cat(new)].double() * w ** 0.5 + pairs[torch.cat(rows)].double()
    x = _rms(x, eps) * _w(case, seed, "embed.norm", w, dtype=f32)
    latents = []
    for i, kind in enumerate(pattern):
        pre = f"l{i}.mix."

        def mat(name, *shape, dtype=torch.bfloat16):
            return _w(case, seed, pre + name, *shape, dtype=dtype)

        def gate(h, name):
            return torch.sigmoid(h @ _w(case, seed, f"l{i}.{name}", w, w).t()
                                 + _w(case, seed, f"l{i}.{name}.b", w, dtype=f32))

        h = _rms(x, eps) * _w(case, seed, f"l{i}.norm1", w, dtype=f32)
        weight = _w(case, seed, f"l{i}.canon1", w, TAPS, dtype=f32)
        rings = _random(seed, f"state{i + 1}.0", (len(new), TAPS - 1, w)).bfloat16()
        u = h + torch.cat([_conv(r, _ring_past(ring, past, TAPS), weight) for r, ring, (past, _)
                           in zip(_split(h, new), rings, portions)])
        if kind == "o":
            own = _rms(u @ mat("dkv", rank, w).t(), eps) * mat("dkv.norm", rank, dtype=f32)
            at = pattern[:i].count("o")
            latents = [torch.cat([c0[:, 0, :rank], c]) for c0, c in zip(
                _contexts(case, seed, at, "k", (1, rank)), _split(own, new))]
        q = (u @ mat("q", H * d, w).t()).view(-1, H, d)
        uk, uv, sink = mat("uk", H * d, rank), mat("uv", H * d, rank), mat("sink", H, dtype=f32)
        a = torch.cat([_attend(r, (c @ uk.t()).view(-1, H, d), (c @ uv.t()).view(-1, H, d), past,
                               d ** -0.5, sink=sink)
                       for r, c, (past, _) in zip(_split(q, new), latents, portions)])
        a = a * torch.sigmoid(u @ mat("g", H, w).t())[:, :, None]
        x = x + gate(h, "rg1") * (a.flatten(1) @ mat("o", w, H * d).t())
        h = _rms(x, eps) * _w(case, seed, f"l{i}.norm2", w, dtype=f32)
        pre = f"l{i}.mlp."
        z = h @ mat("up", ff, w).t()
        p, n = torch.nn.functional.softplus(mat("act", 2, dtype=f32))
        z = torch.where(z > 0, p * z * z, (0.5 + n) * (torch.expm1(z.clamp(max=0)) - z)) + z / 2
        x = x + gate(h, "rg2") * (z @ mat("down", w, ff).t())
    x = _rms(_last(x, new), eps) * _w(case, seed, "final.norm", w, dtype=f32)
    return x @ _w(case, seed, "head", HYBRID_VOCAB, w).t()


def _exact_encode(case, seed):
    texts = [torch.tensor(t, device=DEV) for t in _texts(case, seed)]
    d = 64

    def mat(name, *shape):
        return _w({"model": "senotar-1024"}, seed, name, *shape)

    x = mat("embed.weight", 30522, 768)[torch.cat(texts)]
    pos = torch.cat([torch.arange(len(t), device=DEV) for t in texts])
    for i in range(12):
        pre = f"layers.{i}."
        h = _rms(x, 1e-12) * mat(pre + "norm1", 768)
        q, k, v = (h @ mat(pre + "qkv.weight", 3 * 768, 768).t()).view(-1, 36, d).split(12, 1)
        q, k = _rotate(q, pos, d, 1e4), _rotate(k, pos, d, 1e4)
        outs = []
        for a, b, c in zip(_split(q, texts), _split(k, texts), _split(v, texts)):
            s = torch.softmax(torch.einsum("ihd,jhd->hij", a, b) * d ** -0.5, -1)
            outs.append(torch.einsum("hij,jhd->ihd", s, c))
        x = x + torch.cat(outs).flatten(1) @ mat(pre + "o.weight", 768, 768).t()
        h = _rms(x, 1e-12) * mat(pre + "norm2", 768)
        g, u = (h @ mat(pre + "gate_up.weight", 2 * 3072, 768).t()).chunk(2, -1)
        x = x + (torch.nn.functional.silu(g) * u) @ mat(pre + "down.weight", 768, 3072).t()
    x = _rms(x, 1e-12) * mat("final_norm", 768)
    x = torch.stack([s.mean(0) for s in _split(x, texts)])
    return x / x.norm(dim=-1, keepdim=True)
