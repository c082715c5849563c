"""The work users have this package do, as timed cases.

Five kinds of pass, each through the public entry points a user's program calls:

  decode    one token per sequence through ``Attention.forward`` with a block KV cache: append
            (with rotary embeddings where the model has them) and attention, one layer
  prefill   a chunk of new tokens per sequence through the same call; chunks of equal length
            behind a cached prefix, or prompts of unequal length packed into one step
  dense     ``Attention.forward(query, key, value, attention_mask)``, the call without a cache:
            scoring and evaluation under a causal mask, packed documents under their own mask
  generate  ``generation.generate``: prefill of the prompts, then greedy decode
  step      one decode step of a whole model, ``LanguageModel.forward`` with a KV cache

``listed`` names one case for each use (what it stands for is beside it); ``draw`` spreads the
same kinds over their ranges.  The passes return everything they compute: attention outputs, the
pools the new rows went into, logits, tokens and their margins.
"""
import math

import numpy as np
import torch

from ironcore_amd import generation
from ironcore_amd.config import (InitConfig, MainConfig, ModelConfig, PositionalEmbeddingConfig, TrainerConfig,
                                 gpt2_small_config)
from ironcore_amd.kv_cache import PagedKVCache
from ironcore_amd.layers import Attention, PagedAttentionMetadata, RotaryPositionalEmbedding

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}


def _decode(name, batch, heads, groups, hd, lo, hi, dtype="bf16", block=16, rope=False):
    return {"name": name, "kind": "decode", "batch": batch, "heads": heads, "groups": groups, "hd": hd,
            "ctx_lo": lo, "ctx_hi": hi, "dtype": dtype, "block": block, "rope": rope}


def _prefill(name, n_seqs, heads, groups, hd, prefix_hi, chunk_lo, chunk_hi, dtype="bf16", block=16, rope=False):
    return {"name": name, "kind": "prefill", "n_seqs": n_seqs, "heads": heads, "groups": groups, "hd": hd,
            "prefix_hi": prefix_hi, "chunk_lo": chunk_lo, "chunk_hi": chunk_hi, "dtype": dtype, "block": block,
            "rope": rope}


def _dense(name, batch, heads, groups, hd, seq, mask, dtype="bf16"):
    return {"name": name, "kind": "dense", "batch": batch, "heads": heads, "groups": groups, "hd": hd, "seq": seq,
            "mask": mask, "dtype": dtype}


def listed():
    return [
        # the smallest call there is: a decode step of the GPT-2 small configuration (batch 4 behind
        # prompts of 128 tokens), fp32; launches and host work are all of it
        _decode("decode_gpt2_layer", 4, 12, 12, 64, 128, 192, dtype="fp32"),
        # the headline: Llama-7B layer shape, batch 64
        _decode("decode_llama7b", 64, 32, 32, 128, 512, 4096),
        # grouped queries and long contexts: Llama-70B attention shape, batch 128 (the largest)
        _decode("decode_llama70b_gqa", 128, 64, 8, 128, 1024, 8192),
        # rollouts: 32 prompts x 16 samples that share their prompt's blocks, decoded as cohorts
        {"name": "decode_rollouts", "kind": "cohorts", "prompts": 32, "samples": 16, "heads": 28, "groups": 4,
         "hd": 128, "prefix": 1024, "suffix_hi": 1024, "dtype": "bf16", "block": 16},
        # one user, one long document: a single sequence of 60 001 tokens, fp16, rotary
        _decode("decode_one_long", 1, 32, 8, 128, 60001, 60001, dtype="fp16", rope=True),
        # a busy server of a small model: 233 short conversations, head dim 64, rotary
        _decode("decode_short_contexts", 233, 16, 16, 64, 17, 512, rope=True),
        # long prompts cut into chunks: Llama-7B dims, 16 x 512 new tokens behind up to 4096 cached ones
        _prefill("prefill_chunks", 16, 32, 32, 128, 4096, 512, 512),
        # new conversations arriving together: prompts of unequal length, nothing cached, grouped queries, rotary
        _prefill("prefill_prompts", 9, 28, 4, 128, 0, 3, 701, rope=True),
        # multiple-choice scoring: 20 questions x 4 endings, causal mask, nothing cached
        _dense("dense_scoring", 80, 12, 12, 64, 129, "causal"),
        # evaluation on packed documents: the block-diagonal causal mask of a packed batch
        _dense("dense_documents", 2, 16, 16, 64, 1024, "documents"),
        # end to end: GPT-2 small, fp32, batch 4, 128 prompt tokens, 64 new ones, the decode step as a HIP graph
        {"name": "generate_gpt2", "kind": "generate", "batch": 4, "prompt": 128, "new": 64, "graph": True},
        # a decode step of a larger model: Llama-7B layer dims (four layers of it), RMSNorm, SwiGLU, rotary
        {"name": "step_llama", "kind": "step", "layers": 4, "d_model": 4096, "d_ffn": 11008, "heads": 32, "groups": 32,
         "vocab": 32000, "batch": 16, "ctx_lo": 512, "ctx_hi": 2048, "dtype": "bf16"},
    ]


# ---- drawn cases -------------------------------------------------------------------------------

HEADS = ((12, 12), (16, 16), (32, 32), (8, 8), (8, 1), (16, 4), (32, 8), (28, 4), (64, 8))
MAX_BYTES = 2.4e9
MAX_FLOPS = 2.5e11


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "cohorts", "prefill", "prefill", "dense", "dense", "generate",
                       "step"))
    heads, groups = rng.choice(HEADS)
    hd = rng.choice((64, 128, 128))
    dtype = rng.choice(("bf16", "bf16", "fp16", "fp32"))
    block = rng.choice((16, 16, 16, 32, 48, 64))
    if kind == "decode":
        batch, hi = _log(rng, 1, 300), _log(rng, 32, 60000)
        lo = max(1, int(hi * rng.uniform(0.05, 1.0)))
        while True:
            case = _decode("", batch, heads, groups, hd, lo, hi, dtype, block, rng.random() < 0.5)
            if work(case)["bytes"] <= MAX_BYTES:
                break
            batch, lo, hi = max(1, batch // 2), max(1, lo * 3 // 4), max(1, hi * 3 // 4)
    elif kind == "cohorts":
        heads, groups = rng.choice(((28, 4), (32, 8), (16, 4), (12, 12)))
        prompts, samples = _log(rng, 2, 40), rng.choice((4, 8, 16))
        while True:
            case = {"kind": kind, "prompts": prompts, "samples": samples, "heads": heads, "groups": groups, "hd": hd,
                    "prefix": block * _log(rng, 4, 64), "suffix_hi": _log(rng, 16, 1200),
                    "dtype": rng.choice(("bf16", "fp16")), "block": block}
            if work(case)["bytes"] <= MAX_BYTES / 2:
                break
            prompts = max(1, prompts // 2)
    elif kind == "prefill":
        n, hi = _log(rng, 1, 32), _log(rng, 16, 2048)
        lo = hi if rng.random() < 0.4 else max(1, int(hi * rng.uniform(0.01, 0.9)))
        prefix = 0 if rng.random() < 0.4 else _log(rng, 16, 8192)
        while True:
            case = _prefill("", n, heads, groups, hd, prefix, lo, hi, dtype, block, rng.random() < 0.5)
            if work(case)["flops"] <= (MAX_FLOPS if dtype != "fp32" else MAX_FLOPS / 8):
                break
            n, prefix, lo, hi = max(1, n * 2 // 3), prefix * 3 // 4, max(1, lo * 3 // 4), max(1, hi * 3 // 4)
    elif kind == "dense":
        batch, seq = _log(rng, 1, 100), _log(rng, 17, 2048)
        while True:
            case = _dense("", batch, heads, groups, hd, seq, rng.choice(("causal", "documents", "none")), dtype)
            if work(case)["flops"] <= (MAX_FLOPS if dtype != "fp32" else MAX_FLOPS / 8) and batch * seq * seq <= 6e7:
                break
            batch, seq = max(1, batch * 2 // 3), max(17, seq * 3 // 4)
    elif kind == "generate":
        case = {"kind": kind, "batch": _log(rng, 1, 12), "prompt": _log(rng, 5, 300), "new": _log(rng, 8, 60),
                "graph": rng.random() < 0.6}
        if not case["graph"]:  # the loop without a graph takes longer for each token
            case["new"] = min(case["new"], 24)
        while work(case)["bytes"] > 3.4e10:
            case["new"] = case["new"] * 3 // 4
    else:
        heads, groups = rng.choice(((8, 8), (8, 2), (16, 16), (16, 4), (32, 32), (32, 8)))
        hi = _log(rng, 64, 2048)
        case = {"kind": kind, "layers": rng.choice((2, 3, 4)), "d_model": heads * 128,
                "d_ffn": heads * rng.choice((256, 344, 384)), "heads": heads, "groups": groups, "vocab": 32000,
                "batch": _log(rng, 1, 40), "ctx_lo": max(1, hi // 3), "ctx_hi": hi, "dtype": rng.choice(("bf16", "fp16"))}
        while work(case)["bytes"] > 3.0e9:
            case["batch"] = max(1, case["batch"] // 2)
    case.pop("name", None)
    return case


# ---- what a user's program holds before the call -------------------------------------------------

def _config(heads, groups, hd, dtype):
    return MainConfig(model=ModelConfig(d_model=heads * hd, num_attention_heads=heads, num_attention_groups=groups,
                                        head_dim=hd, dropout_attn=0.0, precision=dtype),
                      trainer=TrainerConfig(use_flash_attn=False))


def _layer(case):
    return Attention(_config(case["heads"], case["groups"], case["hd"], case["dtype"])).to(DEVICE).eval()


def _rope(case, longest):
    return RotaryPositionalEmbedding(case["hd"], max_seq_len=longest).to(DEVICE) if case["rope"] else None


def _randn(shape, dtype, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32).to(dtype)


def _spread(lo, hi, n):
    """n lengths that cover [lo, hi] evenly: a case's lengths are the same for every seed, their order is not."""
    return [lo + int((hi - lo) * (2 * i + 1) / (2 * n) + 0.5) for i in range(n)]


def _chunks(case):
    """(cached prefix, new tokens) of each sequence of a prefill case: both spread evenly, paired by a fixed
    shuffle."""
    n = case["n_seqs"]
    order = np.random.default_rng(n).permutation(n)
    new = _spread(case["chunk_lo"], case["chunk_hi"], n)
    return [(p, new[k]) for p, k in zip(_spread(0, case["prefix_hi"], n), order)]


def _pools(case, n_blocks, seed):
    shape = (n_blocks, case["groups"], case["block"], case["hd"])
    return tuple(_randn(shape, DTYPES[case["dtype"]], seed + k) for k in (1, 2))


def _tables(n_blocks, perm, first=0):
    """int32 [n, longest] block tables on the host: each row the next blocks of the permuted pool."""
    ends = first + np.cumsum(n_blocks)
    tables = np.zeros((len(n_blocks), max(n_blocks)), dtype=np.int32)
    for row, n, end in zip(tables, n_blocks, ends):
        row[:n] = perm[end - n:end]
    return tables


def _cached_decode(case, seed, tables, ctx, pools, rope=None, cohort=1, shared=None):
    """One decode step of one layer: a sequence's new token is the last of its context."""
    b, hn, gn, hd, dtype = len(ctx), case["heads"], case["groups"], case["hd"], DTYPES[case["dtype"]]
    last = np.asarray(ctx) - 1
    slots = tables[np.arange(b), last // case["block"]].astype(np.int64) * case["block"] + last % case["block"]
    meta = PagedAttentionMetadata(
        block_tables=torch.from_numpy(tables).to(DEVICE),
        context_lens=torch.tensor(ctx, dtype=torch.int32, device=DEVICE),
        slot_mapping=torch.from_numpy(slots).to(DEVICE), max_context_len=max(ctx), cohort_size=cohort,
        cohort_shared_blocks=shared, positions=torch.from_numpy(last.astype(np.int32)).to(DEVICE))
    return {"kind": "attention", "layer": _layer(case), "query": _randn((b, 1, hn, hd), dtype, seed + 3),
            "key": _randn((b, 1, gn, hd), dtype, seed + 4), "value": _randn((b, 1, gn, hd), dtype, seed + 5),
            "mask": None, "kw": {"kv_cache": pools, "attn_metadata": meta, "rotary_pos_emb": rope}}


def _prepare_decode(case, seed):
    rng = np.random.default_rng(seed)
    ctx = [int(n) for n in rng.permutation(_spread(case["ctx_lo"], case["ctx_hi"], case["batch"]))]
    n_blocks = [-(-n // case["block"]) for n in ctx]
    tables = _tables(n_blocks, rng.permutation(sum(n_blocks)))
    return _cached_decode(case, seed, tables, ctx, _pools(case, sum(n_blocks), seed), _rope(case, case["ctx_hi"]))


def _prepare_cohorts(case, seed):
    rng = np.random.default_rng(seed)
    prompts, samples, bs = case["prompts"], case["samples"], case["block"]
    shared = case["prefix"] // bs
    own = rng.permutation(_spread(1, case["suffix_hi"], prompts * samples))
    n_blocks = [-(-int(n) // bs) for n in own]
    total = prompts * shared + sum(n_blocks)
    perm = rng.permutation(total)
    prefix = np.repeat(perm[:prompts * shared].reshape(prompts, shared), samples, axis=0)
    tables = np.concatenate([prefix.astype(np.int32), _tables(n_blocks, perm, prompts * shared)], axis=1)
    return _cached_decode(case, seed, tables, [case["prefix"] + int(n) for n in own], _pools(case, total, seed),
                          cohort=samples,
                          shared=torch.full((prompts,), shared, dtype=torch.int32, device=DEVICE))


def _prepare_prefill(case, seed):
    rng = np.random.default_rng(seed)
    n, hn, gn, hd, bs, dtype = (case[k] for k in ("n_seqs", "heads", "groups", "hd", "block", "dtype"))
    seqs = [_chunks(case)[k] for k in rng.permutation(n)]
    n_blocks = [-(-(p + c) // bs) for p, c in seqs]
    tables = _tables(n_blocks, rng.permutation(sum(n_blocks)))
    width = max(c for _, c in seqs)
    slots, positions = np.full((n, width), -1, dtype=np.int64), np.zeros((n, width), dtype=np.int32)
    for i, (p, c) in enumerate(seqs):
        at = np.arange(p, p + c)
        slots[i, :c] = tables[i, at // bs].astype(np.int64) * bs + at % bs
        positions[i, :c] = at
    cu = rows = None
    if any(c != width for _, c in seqs):
        cu = torch.tensor([0] + list(np.cumsum([c for _, c in seqs])), dtype=torch.int32, device=DEVICE)
        rows = torch.from_numpy(np.flatnonzero(slots >= 0)).to(DEVICE)
    ctx = [p + c for p, c in seqs]
    meta = PagedAttentionMetadata(
        block_tables=torch.from_numpy(tables).to(DEVICE),
        context_lens=torch.tensor(ctx, dtype=torch.int32, device=DEVICE),
        slot_mapping=torch.from_numpy(slots.reshape(-1)).to(DEVICE), max_context_len=max(ctx), cu_seqlens_q=cu,
        positions=torch.from_numpy(positions.reshape(-1)).to(DEVICE), chunk_rows=rows, max_chunk_len=width)
    return {"kind": "attention", "layer": _layer(case), "query": _randn((n, width, hn, hd), DTYPES[dtype], seed + 3),
            "key": _randn((n, width, gn, hd), DTYPES[dtype], seed + 4),
            "value": _randn((n, width, gn, hd), DTYPES[dtype], seed + 5), "mask": None,
            "kw": {"kv_cache": _pools(case, sum(n_blocks), seed), "attn_metadata": meta,
                   "rotary_pos_emb": _rope(case, max(ctx))}}


def _document_mask(batch, seq, seed):
    """[batch, 1, seq, seq], True = visible: packed documents of about an eighth of the row, each causal."""
    rng = np.random.default_rng(seed)
    doc = np.zeros((batch, seq), dtype=np.int64)
    for row in doc:
        for cut in rng.integers(1, max(seq, 2), size=7):
            row[cut:] += 1
    doc = torch.from_numpy(doc).to(DEVICE)
    causal = torch.ones(seq, seq, dtype=torch.bool, device=DEVICE).tril()
    return ((doc.unsqueeze(2) == doc.unsqueeze(1)) & causal).unsqueeze(1)


def _prepare_dense(case, seed):
    b, s, hn, gn, hd = (case[k] for k in ("batch", "seq", "heads", "groups", "hd"))
    dtype = DTYPES[case["dtype"]]
    mask = None
    if case["mask"] == "causal":
        mask = torch.tril(torch.ones(s, s, device=DEVICE)).view(1, 1, s, s) > 0.5
    elif case["mask"] == "documents":
        mask = _document_mask(b, s, seed)
    return {"kind": "attention", "layer": _layer(case), "query": _randn((b, s, hn, hd), dtype, seed + 1),
            "key": _randn((b, s, gn, hd), dtype, seed + 2), "value": _randn((b, s, gn, hd), dtype, seed + 3),
            "mask": mask, "kw": {}}


def _model(config, vocab, dtype, seed):
    torch.manual_seed(seed)
    with torch.device(DEVICE):
        return generation.LanguageModel(config, vocab_size=vocab).to(dtype).eval()


def _tokens(shape, vocab, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return torch.randint(0, vocab, shape, generator=g, device=DEVICE)


def _prepare_generate(case, seed):
    return {"kind": "generate", "model": _model(gpt2_small_config("fp32"), 50257, torch.float32, seed),
            "ids": _tokens((case["batch"], case["prompt"]), 50257, seed + 1), "new": case["new"],
            "graph": case["graph"]}


def _prepare_step(case, seed):
    """A model whose sequences sit in its cache, one new token each."""
    hd, dtype = case["d_model"] // case["heads"], DTYPES[case["dtype"]]
    longest = case["ctx_hi"] + 1
    config = MainConfig(
        model=ModelConfig(d_model=case["d_model"], d_ffn=case["d_ffn"], num_layers=case["layers"],
                          num_attention_heads=case["heads"], num_attention_groups=case["groups"], head_dim=hd,
                          max_seq_len=longest, max_position_embeddings=longest, dropout_embd=0.0, dropout_attn=0.0,
                          dropout_mlp=0.0, precision=case["dtype"], untie_embed=True, no_bias=True,
                          ln_type="rmsnorm", activation_type="swiglu",
                          positional_embedding=PositionalEmbeddingConfig(type="rope")),
        trainer=TrainerConfig(use_flash_attn=False), init=InitConfig(seed=0, init_std=0.02))
    model = _model(config, case["vocab"], dtype, seed)
    b = case["batch"]
    past = np.random.default_rng(seed).permutation(_spread(case["ctx_lo"], case["ctx_hi"], b))
    blocks = int(sum((n + 1 + 15) // 16 for n in past))
    cache = PagedKVCache(case["layers"], blocks, 16, case["groups"], hd, dtype, DEVICE)
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed + 2)
    cache.k_pools.normal_(generator=g)
    cache.v_pools.normal_(generator=g)
    ids = [cache.add_sequence() for _ in range(b)]
    for sid, n in zip(ids, past):
        cache.reserve(sid, int(n))
        cache.advance([sid], int(n))
    return {"kind": "step", "model": model, "cache": cache, "meta": cache.prepare(ids, 1),
            "ids": _tokens((b, 1), case["vocab"], seed + 3),
            "positions": torch.from_numpy(past).to(DEVICE).unsqueeze(1)}


def prepare(case, seed):
    return {"decode": _prepare_decode, "cohorts": _prepare_cohorts, "prefill": _prepare_prefill,
            "dense": _prepare_dense, "generate": _prepare_generate, "step": _prepare_step}[case["kind"]](case, seed)


# ---- one pass --------------------------------------------------------------------------------------

@torch.no_grad()
def run(state):
    if state["kind"] == "attention":
        out = state["layer"](state["query"], state["key"], state["value"], state["mask"], **state["kw"])
        if "kv_cache" in state["kw"]:
            return (out,) + tuple(state["kw"]["kv_cache"])
        return out
    if state["kind"] == "generate":
        tokens, margins = generation.generate(state["model"], state["ids"], state["new"], return_margins=True,
                                              use_graph=state["graph"])
        return tokens, margins
    logits = state["model"](state["ids"], kv_cache=state["cache"], attn_metadata=state["meta"],
                            position_ids=state["positions"])
    return logits, state["cache"].k_pools, state["cache"].v_pools


# ---- what a pass cannot do without -----------------------------------------------------------------

def work(case):
    """Bytes: inputs read once (K and V rows once for all that see them), outputs written once.
    Flops: two per multiply-add, visible (query, key) pairs only."""
    kind = case["kind"]
    if kind == "generate":
        # prefill once, then one pass over the weights (12 layers of d_model 768 and the vocabulary) a step
        weights = 12 * (12 * 768 * 768) + 50304 * 768
        b, n = case["batch"], case["new"]
        ctx = b * (case["prompt"] + n / 2)
        return {"bytes": 4 * n * (weights + 12 * 2 * 768 * ctx),
                "flops": 2 * weights * b * n + 2 * 12 * 12 * 768 * 768 * b * case["prompt"]}
    size, hn, gn = SIZES[case["dtype"]], case["heads"], case["groups"]
    if kind == "step":
        d, b, hd = case["d_model"], case["batch"], case["d_model"] // hn
        weights = case["layers"] * (2 * d * d + 2 * d * gn * hd + 3 * d * case["d_ffn"]) + case["vocab"] * d
        tokens = case["layers"] * (sum(_spread(case["ctx_lo"], case["ctx_hi"], b)) + b)
        return {"bytes": size * (weights + tokens * 2 * gn * hd + b * case["vocab"]),
                "flops": 2 * weights * b + 4 * hn * hd * tokens}
    hd = case["hd"]
    if kind in ("decode", "cohorts"):
        if kind == "decode":
            b = case["batch"]
            seen = stored = sum(_spread(case["ctx_lo"], case["ctx_hi"], b))
        else:
            b, prefix = case["prompts"] * case["samples"], case["prefix"]
            own = sum(_spread(1, case["suffix_hi"], b))
            seen, stored = b * prefix + own, case["prompts"] * prefix + own
        return {"bytes": size * (stored * 2 * gn * hd + b * (2 * hn + 4 * gn) * hd) + 4 * seen / case["block"],
                "flops": 4 * hn * hd * seen}
    if kind == "prefill":
        seqs = _chunks(case)
        new = sum(c for _, c in seqs)
        return {"bytes": size * hd * ((new + sum(p for p, _ in seqs)) * 2 * gn + new * (2 * hn + 4 * gn)),
                "flops": 4 * hn * hd * sum(c * p + c * (c + 1) / 2 for p, c in seqs)}
    b, s = case["batch"], case["seq"]
    # a row in eight random pieces: on average the squares of their lengths sum to 2/9 of its square
    pairs = {"none": s * s, "causal": s * (s + 1) / 2, "documents": (s * s * 2 / 9 + s) / 2}[case["mask"]]
    mask = {"none": 0, "causal": s * s, "documents": b * s * s}[case["mask"]]
    return {"bytes": size * hd * b * s * (2 * hn + 2 * gn) + mask, "flops": 4 * hn * hd * b * pairs}


def tolerance(case):
    """About four times the distance seen to the same pass in float64 (attention: 2.4e-3, 3.0e-4 and 1.7e-7 in
    bf16, fp16 and fp32; margins: 2.9e-6) or, for a whole 16-bit model, to the pass in fp32 (bf16: 1.5e-2, twice
    that stated)."""
    if case["kind"] == "generate":
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.0}
    if case["kind"] == "step":
        return {"rel": 3e-2, "max": 0.3} if case["dtype"] == "bf16" else {"rel": 6e-3, "max": 6e-2}
    return {"bf16": {"rel": 1e-2, "max": 5e-2}, "fp16": {"rel": 1.2e-3, "max": 8e-3},
            "fp32": {"rel": 2e-6, "max": 2e-5}}[case["dtype"]]
