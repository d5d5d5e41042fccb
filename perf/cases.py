"""What a user of these operators has them do, as timed cases.

A serving engine calls the operators of ``dlcompiler_amd`` once per decoder layer and step, so the
cases are the calls of such a step, at the sizes a step has in earnest:

* ``layer``    the row operators around the engine's own GEMMs: residual add + RMSNorm before and
               after the attention, rotary embedding, KV-cache fill, SiLU-and-mul
* ``gate``     the MoE router: softmax, top-k, renormalisation and expert alignment
* ``prefill``  causal attention over packed prompts
* ``chunked``  attention of prompt chunks over the paged history they continue
* ``decode``   paged attention of one new token per sequence
* ``moe``      the reference's fused MoE MLP: 16-bit row-major weights, routing given
* ``moe_fp8``  the fp8 MoE layer from the router's logits, weights laid out once at load time

Small sizes are decode steps of a few sequences, where latency and launches count; large ones are
prompt batches.  Sizes of the large cases are the benchmark configurations of ``bench.py``.
"""
import math
import random

import torch

from dlcompiler_amd.kernels.activation import silu_and_mul
from dlcompiler_amd.kernels.apply_rotary_pos_emb import apply_rotary_pos_emb
from dlcompiler_amd.kernels.fill_kv_cache import fill_kv_cache
from dlcompiler_amd.kernels.fused_moe import ALIGN_BLOCK, fused_moe, fused_moe_fp8, shuffle_moe_weight
from dlcompiler_amd.kernels.moe_gating import moe_topk_softmax_align
from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd
from dlcompiler_amd.kernels.prefill_attention import context_attention_fwd
from dlcompiler_amd.kernels.rms_norm import add_rms_norm

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE_OF = {"bf16": 2, "fp16": 2, "fp32": 4}

# Ceilings of a drawn case: what the largest listed cases take.
MOST_MOE_FLOPS = 3.9e11
MOST_ATTENTION_FLOPS = 2.2e11
MOST_KV_BYTES = 1.0e9
MOST_MOE_WEIGHTS = 5.5e8


def listed():
    attn = {"heads": 32, "kv_heads": 8, "head_dim": 128, "dtype": "bf16"}
    mlp = {"hidden": 2048, "inter": 1408, "experts": 64, "topk": 6, "local": 64, "offset": 0, "dtype": "bf16"}
    layer = {"hidden": 4096, "inter": 11008, "page": 64, **attn}
    return [
        # one decode step of eight sequences: five small launches behind each other
        {"name": "layer_decode_8", "op": "layer", "seqs": 8, "lo": 1, "hi": 1, "history": 1500, "mix": 1, **layer},
        # a prompt batch: every operator is a stream through memory
        {"name": "layer_prefill_16k", "op": "layer", "seqs": 8, "lo": 512, "hi": 3584, "history": 0, "mix": 2,
         **layer},
        # router of a decode step; engines keep its logits in 16 bits
        {"name": "gate_decode_48", "op": "gate", "tokens": 48, "experts": 64, "topk": 6, "block": 128,
         "dtype": "bf16"},
        # router of a prompt batch
        {"name": "gate_prefill_16k", "op": "gate", "tokens": 16384, "experts": 64, "topk": 6, "block": 64,
         "dtype": "fp32"},
        # a few short prompts, small head size: too little work to fill the chip
        {"name": "prefill_short", "op": "prefill", "seqs": 3, "lo": 33, "hi": 700, "mix": 3, "heads": 16,
         "kv_heads": 4, "head_dim": 64, "dtype": "fp16", "index64": True},
        # a full prompt batch
        {"name": "prefill_8x4096", "op": "prefill", "seqs": 8, "lo": 512, "hi": 4096, "mix": 4, "index64": False,
         **attn},
        # chunked prefill: the next 300 to 600 tokens of each sequence over its history
        {"name": "chunked_8x512", "op": "chunked", "seqs": 8, "lo": 300, "hi": 600, "history": 4096, "mix": 5,
         "page": 64, "window": 0, "softcap": 0.0, "index64": True, **attn},
        # one user's decode step
        {"name": "decode_1x4000", "op": "decode", "seqs": 1, "lo": 4000, "hi": 4000, "mix": 6, "page": 64,
         "window": 0, "softcap": 0.0, "index64": True, **attn},
        # a full decode batch
        {"name": "decode_64x8192", "op": "decode", "seqs": 64, "lo": 512, "hi": 8192, "mix": 7, "page": 64,
         "window": 0, "softcap": 0.0, "index64": False, **attn},
        # MoE layer of a decode step: a few rows per expert, bound by reading the experts' weights
        {"name": "moe_fp8_decode_32", "op": "moe_fp8", "tokens": 32, **mlp},
        # MoE layer of a prompt batch: bound by the matrix cores
        {"name": "moe_fp8_prefill_4096", "op": "moe_fp8", "tokens": 4096, **mlp},
        # the reference's own operator at a busy mixed step
        {"name": "moe_bf16_300", "op": "moe", "tokens": 300, "renormalize": True, **mlp},
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_heads(rng):
    heads, kv_heads = rng.choice([(32, 8), (32, 8), (16, 4), (28, 4), (40, 8), (64, 8), (16, 16), (8, 1)])
    return {"heads": heads, "kv_heads": kv_heads, "head_dim": rng.choice([128, 128, 128, 64, 64, 96]),
            "dtype": rng.choice(["bf16", "bf16", "fp16"])}


def _draw_options(rng):
    """Sliding window and soft-cap are options of some models only."""
    return {"window": rng.choice([0, 0, 0, 1024]), "softcap": rng.choice([0.0, 0.0, 0.0, 30.0]),
            "page": rng.choice([16, 32, 64, 64, 128]), "index64": rng.random() < 0.5}


def _draw_layer(rng):
    case = {"op": "layer", "hidden": 128 * _log_uniform(rng, 8, 64), "inter": 64 * _log_uniform(rng, 16, 224),
            "page": rng.choice([16, 64, 128]), "mix": rng.randrange(1000), **_draw_heads(rng)}
    if rng.random() < 0.5:
        case.update(seqs=_log_uniform(rng, 1, 256), lo=1, hi=1, history=_log_uniform(rng, 64, 2048))
    else:
        hi = _log_uniform(rng, 32, 4096)
        case.update(seqs=rng.randint(1, max(1, min(16, 16384 // hi))), lo=max(1, hi // 8), hi=hi, history=0)
    return case


def _draw_gate(rng):
    experts, topk = rng.choice([(8, 2), (16, 2), (60, 4), (64, 6), (64, 8), (128, 8), (256, 8)])
    return {"op": "gate", "tokens": _log_uniform(rng, 1, 16384), "experts": experts, "topk": topk,
            "block": rng.choice([16, 64, 128, 128]), "dtype": rng.choice(["fp32", "fp32", "bf16", "fp16"])}


def _draw_prefill(rng):
    case = {"op": "prefill", "mix": rng.randrange(1000), "index64": rng.random() < 0.5, **_draw_heads(rng)}
    case["hi"] = _log_uniform(rng, 16, 8192)
    case["lo"] = max(1, case["hi"] // rng.choice([1, 4, 16]))
    case["seqs"] = _log_uniform(rng, 1, 16)
    while case["seqs"] > 1 and _attention_flops(case) > MOST_ATTENTION_FLOPS:
        case["seqs"] -= 1
    while _attention_flops(case) > MOST_ATTENTION_FLOPS:
        case["hi"] = case["hi"] * 3 // 4
        case["lo"] = min(case["lo"], case["hi"])
    return case


def _draw_chunked(rng):
    case = {"op": "chunked", "mix": rng.randrange(1000), **_draw_heads(rng), **_draw_options(rng)}
    case["hi"] = _log_uniform(rng, 16, 2048)
    case["lo"] = max(2, case["hi"] // rng.choice([1, 4, 16]))
    case["history"] = _log_uniform(rng, 32, 16384)
    case["seqs"] = _log_uniform(rng, 1, 16)
    while _attention_flops(dict(case, window=0)) > MOST_ATTENTION_FLOPS:
        if case["seqs"] > 1:
            case["seqs"] -= 1
        else:
            case["history"] = case["history"] * 3 // 4
    return case


def _draw_decode(rng):
    case = {"op": "decode", "mix": rng.randrange(1000), **_draw_heads(rng), **_draw_options(rng)}
    case["hi"] = _log_uniform(rng, 64, 32768)
    case["lo"] = max(1, case["hi"] // rng.choice([1, 4, 16]))
    case["seqs"] = _log_uniform(rng, 1, 256)
    while case["seqs"] > 1 and case["seqs"] * case["hi"] * case["kv_heads"] * case["head_dim"] * 4 > MOST_KV_BYTES:
        case["seqs"] = max(1, case["seqs"] * 3 // 4)
    return case


def _draw_moe(rng):
    op = rng.choice(["moe", "moe_fp8", "moe_fp8"])
    experts, topk = rng.choice([(8, 2), (16, 4), (32, 4), (64, 6), (64, 6), (64, 8), (128, 8)])
    case = {"op": op, "experts": experts, "topk": topk, "local": experts, "offset": 0,
            "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if rng.random() < 0.2:  # one rank of an expert-parallel group
        case["local"] = experts // 2
        case["offset"] = rng.choice([0, experts // 2])
    case["hidden"] = 128 * _log_uniform(rng, 8, 32)
    case["inter"] = 128 * _log_uniform(rng, 2, 32)
    while 3 * case["local"] * case["hidden"] * case["inter"] > MOST_MOE_WEIGHTS:
        case["inter"] = max(128, case["inter"] // 256 * 128)
    case["tokens"] = _log_uniform(rng, 1, 4096)
    limit = MOST_MOE_FLOPS if op == "moe_fp8" else MOST_MOE_FLOPS / 2
    while work(case)["flops"] > limit:
        case["tokens"] = case["tokens"] * 3 // 4
    if op == "moe":
        case["renormalize"] = rng.random() < 0.5
    return case


def draw(rng):
    return rng.choice([_draw_layer, _draw_layer, _draw_gate, _draw_gate, _draw_prefill, _draw_chunked,
                       _draw_decode, _draw_decode, _draw_moe, _draw_moe, _draw_moe])(rng)


# --------------------------------------------------------------------------------------
# shapes that follow from a case alone
# --------------------------------------------------------------------------------------
def _lengths(case):
    """New tokens (for ``decode``: context lengths) of each sequence, uniform in [lo, hi]."""
    rng = random.Random(case["mix"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["seqs"])]


def _histories(case):
    """Cached tokens of each sequence ahead of the new ones."""
    if not case.get("history"):
        return [0] * case["seqs"]
    rng = random.Random(case["mix"] + 1)
    return [rng.randint(case["history"] // 8, case["history"]) for _ in range(case["seqs"])]


def _visible(new, history, window):
    """(query, key) pairs that causal attention of ``new`` tokens over ``history`` looks at."""
    pairs = 0
    for i in range(new):
        keys = history + i + 1
        pairs += min(keys, window + 1) if window else keys
    return pairs


def _attention_flops(case):
    if case["op"] == "decode":
        span = case["window"] + 1 if case["window"] else case["hi"]
        pairs = sum(min(n, span) for n in _lengths(case))
    elif case.get("window"):
        pairs = sum(_visible(n, h, case["window"]) for n, h in zip(_lengths(case), _histories(case)))
    else:
        pairs = sum(n * h + n * (n + 1) // 2 for n, h in zip(_lengths(case), _histories(case)))
    return 4.0 * case["head_dim"] * case["heads"] * pairs


def work(case):
    op, size = case["op"], SIZE_OF[case["dtype"]]
    if op == "gate":
        slots = case["tokens"] * case["topk"]
        padded = slots + min(case["experts"], slots) * (case["block"] - 1) // 2
        words = 3 * slots + padded + padded // case["block"] + case["experts"]
        return {"bytes": case["tokens"] * case["experts"] * size + 4 * words,
                "flops": case["tokens"] * case["experts"] * (4 + case["topk"])}
    if op in ("moe", "moe_fp8"):
        slots = case["tokens"] * case["topk"] * case["local"] / case["experts"]
        hit = case["local"] * (1.0 - (1.0 - case["topk"] / case["experts"]) ** case["tokens"])
        weights = hit * 3 * case["hidden"] * case["inter"] * (1 if op == "moe_fp8" else size)
        rows = 2 * case["tokens"] * case["hidden"] * size
        routing = case["tokens"] * (case["experts"] * 4 if op == "moe_fp8" else case["topk"] * 12)
        return {"bytes": weights + rows + routing, "flops": 6.0 * slots * case["hidden"] * case["inter"]}
    lengths = _lengths(case)
    head_row = case["head_dim"] * size
    if op == "layer":
        tokens = sum(lengths)
        norms = 2 * 4 * tokens * case["hidden"] * size
        rotary = 2 * tokens * (case["heads"] + case["kv_heads"]) * head_row + 2 * tokens * head_row
        fill = 4 * tokens * case["kv_heads"] * head_row
        act = 3 * tokens * case["inter"] * size
        return {"bytes": norms + rotary + fill + act,
                "flops": tokens * (16.0 * case["hidden"] + 3.0 * (case["heads"] + case["kv_heads"])
                                   * case["head_dim"] + 6.0 * case["inter"])}
    if op == "decode":
        span = case["window"] + 1 if case["window"] else case["hi"]
        kv_rows = sum(min(n, span) for n in lengths)
        q_rows = case["seqs"]
    else:
        # keys that no query of the sequence sees (older than the window of its first query) count out
        window = case.get("window") or 0
        kv_rows = sum(n + (min(h, window) if window else h) for n, h in zip(lengths, _histories(case)))
        q_rows = sum(lengths)
    return {"bytes": 2 * kv_rows * case["kv_heads"] * head_row + 2 * q_rows * case["heads"] * head_row,
            "flops": _attention_flops(case)}


def tolerance(case):
    if case["op"] == "gate":
        return {"rel": 1e-5}  # fp32 weights; ids, sorted slots, block experts and counts are whole numbers
    return {"rel": 1e-2 if case["dtype"] == "bf16" or case["op"] == "moe_fp8" else 2e-3}


# --------------------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------------------
def _starts(lengths):
    return [sum(lengths[:i]) for i in range(len(lengths))]


def _paged_cache(case, context, gen, normal):
    """K and V caches whose pages belong to the sequences in random order, and the block table."""
    page, dev = case["page"], gen.device
    blocks = [-(-n // page) for n in context]
    pages = torch.randperm(sum(blocks), generator=gen, device=dev)
    table = torch.zeros((len(context), max(blocks)), dtype=torch.int64, device=dev)
    at = 0
    for i, n in enumerate(blocks):
        table[i, :n] = pages[at:at + n]
        at += n
    shape = (sum(blocks), page, case["kv_heads"], case["head_dim"])
    return normal(*shape), normal(*shape), table


def _block_quantised(w):
    """fp8 weights with one fp32 scale per 128 x 128 block."""
    experts, rows, cols = w.shape
    blocks = w.view(experts, rows // 128, 128, cols // 128, 128)
    scale = blocks.abs().amax(dim=(2, 4)).float().clamp_min(1e-10) / 448.0
    scaled = blocks / scale[:, :, None, :, None]
    return scaled.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(experts, rows, cols), scale


def prepare(case, seed):
    dev, dtype, op = torch.device("cuda"), DTYPES[case["dtype"]], case["op"]
    gen = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape, std=1.0, as_type=dtype):
        return torch.randn(shape, generator=gen, device=dev, dtype=as_type) * std

    def index(values):
        return torch.tensor(values, dtype=torch.int64 if case.get("index64") else torch.int32, device=dev)

    state = {"case": case}
    if op == "gate":
        state["logits"] = normal(case["tokens"], case["experts"])
    elif op in ("moe", "moe_fp8"):
        tokens, hidden, inter, local = case["tokens"], case["hidden"], case["inter"], case["local"]
        state["x"] = normal(tokens, hidden)
        logits = normal(tokens, case["experts"], as_type=torch.float32)
        gate_up, down = normal(local, 2 * inter, hidden, std=0.02), normal(local, hidden, inter, std=0.02)
        if op == "moe":
            state["w1"], state["w2"] = gate_up, down
            state["weights"], state["ids"] = torch.topk(torch.softmax(logits, -1), case["topk"], dim=-1)
        else:
            state["logits"] = logits
            w1, state["s1"] = _block_quantised(gate_up)
            w2, state["s2"] = _block_quantised(down)
            state["w1"], state["w2"] = shuffle_moe_weight(w1), shuffle_moe_weight(w2)
    elif op == "layer":
        lengths, histories = _lengths(case), _histories(case)
        tokens, heads, kv_heads, dim = sum(lengths), case["heads"], case["kv_heads"], case["head_dim"]
        context = [n + h for n, h in zip(lengths, histories)]
        state["hidden"], state["residual"] = normal(tokens, case["hidden"]), normal(tokens, case["hidden"])
        state["norm1"] = 1.0 + normal(case["hidden"], std=0.1)
        state["norm2"] = 1.0 + normal(case["hidden"], std=0.1)
        state["q"], state["k"], state["v"] = (normal(tokens, n, dim) for n in (heads, kv_heads, kv_heads))
        state["q_embed"], state["k_embed"] = torch.empty_like(state["q"]), torch.empty_like(state["k"])
        position = torch.cat([torch.arange(h, h + n, device=dev) for n, h in zip(lengths, histories)])
        speed = 10000.0 ** (-torch.arange(0, dim, 2, device=dev) / dim)
        angle = (position[:, None] * speed).repeat(1, 2)
        state["cos"], state["sin"] = angle.cos().to(dtype), angle.sin().to(dtype)
        state["k_cache"], state["v_cache"], state["table"] = _paged_cache(case, context, gen, normal)
        state["start"], state["new"], state["context"] = index(_starts(lengths)), index(lengths), index(context)
        state["longest"] = max(lengths)
        state["gate_up"] = normal(tokens, 2 * case["inter"])
    elif op == "decode":
        context = _lengths(case)
        state["q"] = normal(case["seqs"], case["heads"], case["head_dim"])
        state["k"], state["v"], table = _paged_cache(case, context, gen, normal)
        state["table"] = table if case["index64"] else table.to(torch.int32)
        state["start"], state["new"] = index(range(case["seqs"])), index([1] * case["seqs"])
        state["context"], state["longest"] = index(context), 1
        state["out"] = torch.empty_like(state["q"])
    elif op == "chunked":
        lengths = _lengths(case)
        context = [n + h for n, h in zip(lengths, _histories(case))]
        state["q"] = normal(sum(lengths), case["heads"], case["head_dim"])
        state["k"], state["v"], table = _paged_cache(case, context, gen, normal)
        state["table"] = table if case["index64"] else table.to(torch.int32)
        state["start"], state["new"] = index(_starts(lengths)), index(lengths)
        state["context"], state["longest"] = index(context), max(lengths)
        state["out"] = torch.empty_like(state["q"])
    else:
        lengths = _lengths(case)
        tokens, dim = sum(lengths), case["head_dim"]
        state["q"] = normal(tokens, case["heads"], dim)
        state["k"], state["v"] = normal(tokens, case["kv_heads"], dim), normal(tokens, case["kv_heads"], dim)
        state["start"], state["new"], state["longest"] = index(_starts(lengths)), index(lengths), max(lengths)
        state["out"] = torch.empty_like(state["q"])
    return state


# --------------------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------------------
def run(state):
    s, case = state, state["case"]
    op = case["op"]
    if op == "layer":
        normed, residual = add_rms_norm(s["hidden"], s["norm1"], 1e-6, s["residual"])
        apply_rotary_pos_emb(s["q"], s["k"], s["cos"], s["sin"], s["q_embed"], s["k_embed"])
        fill_kv_cache(s["k_embed"], s["v"], s["k_cache"], s["v_cache"], s["start"], s["new"], s["context"],
                      s["longest"], s["table"])
        normed2, residual2 = add_rms_norm(normed, s["norm2"], 1e-6, residual)
        act = silu_and_mul(s["gate_up"])
        return [normed, residual, s["q_embed"], s["k_embed"], s["k_cache"], s["v_cache"], normed2, residual2, act]
    if op == "gate":
        return moe_topk_softmax_align(s["logits"], case["topk"], case["block"], return_counts=True)
    if op == "prefill":
        context_attention_fwd(s["q"], s["k"], s["v"], s["out"], s["start"], s["new"], s["longest"])
        return s["out"]
    if op in ("chunked", "decode"):
        paged_attention_fwd(s["q"], s["k"], s["v"], s["out"], s["table"], s["start"], s["new"], s["context"],
                            s["longest"], window_size=case["window"] or None,
                            logit_softcapping=case["softcap"] or None)
        return s["out"]
    if op == "moe":
        return fused_moe(s["x"], s["w1"], s["w2"], s["weights"], s["ids"], case["topk"], case["offset"],
                         case["experts"], case["renormalize"])
    weights, ids, slots, _, _, counts = moe_topk_softmax_align(s["logits"], case["topk"], ALIGN_BLOCK,
                                                               return_counts=True)
    return fused_moe_fp8(s["x"], s["w1"], s["s1"], s["w2"], s["s2"], weights, ids, case["topk"], case["offset"],
                         case["experts"], weights_shuffled=True, alignment=(slots, counts))
