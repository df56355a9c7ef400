"""Performance cases of the MI355X decode path: what a serving program asks of it.

Five families, each through the package's public entry points:

  decode  FP8 paged-attention decode (`pa_decode_ps_launch`): 16- and
          64-token pages with a block table, sliding windows, and the
          1024-token pages of the work-list route (`get_pa_metadata`)
  layer   the attention part of one decode layer: the KV-cache writer
          (NeoX RoPE, fp8 quantisation, paged scatter) for the new tokens,
          then the paged decode over the cache it wrote to
  rope    the KV-cache writer alone, over prefill and decode token counts
  qknr    fused RMSNorm + GPT-J RoPE + fp8 quantisation of Q and the KV row
  mla     MLA fp8 decode over its work list, then the reduce of cut rows

Inputs are seeded and made on the GPU.  Context lengths belong to the case
(drawn from its `lengths` seed), so a case's bytes do not depend on the
seed of its values.
"""

import math

import numpy as np
import torch

from flydsl_amd import (
    build_fused_rope_cache_module,
    flydsl_mla_fwd_decode,
    flydsl_qk_norm_rope_quant,
    get_mla_metadata_info_v1,
    get_mla_metadata_v1,
    get_pa_metadata,
    get_recommended_splits,
    mla_reduce_v1,
    pa_decode_ps_launch,
)

FP8 = torch.float8_e4m3fn
FP8_MAX = 448.0
MAX_POS = 8192  # rows of the cos/sin tables


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------


def _decode(name, batch, ql, heads, kv_heads, page, ctx, *, head=128, per_token=False, window=0, dtype="bf16",
            lengths=7):
    c = {"family": "decode", "batch": batch, "ql": ql, "heads": heads, "kv_heads": kv_heads, "page": page,
         "ctx": ctx, "head": head, "per_token": per_token, "window": window, "dtype": dtype, "lengths": lengths}
    return dict(c, name=name) if name else c


def listed():
    return [
        # A small batch of short chats: one layer's cache write and decode,
        # where launches and host work count.
        {"name": "layer_small", "family": "layer", "batch": 4, "heads": 8, "kv_heads": 2, "page": 16,
         "ctx": "uniform:1:512", "lengths": 7},
        # The Llama-3-8B-shaped decode step: every sequence at 4096 tokens.
        _decode("decode_llama8b", 64, 1, 32, 8, 16, "fixed:4096"),
        # A serving batch of very different context lengths, per-token scales.
        _decode("decode_ragged", 128, 1, 32, 8, 16, "lognormal:2048:1.0:16:32768", per_token=True),
        # Sliding-window layers over long contexts.
        _decode("decode_window", 32, 1, 32, 8, 16, "uniform:8192:32768", window=4096),
        # Speculative decode: four query tokens per sequence, 64-token pages.
        _decode("decode_mtp", 256, 4, 64, 4, 64, "uniform:4096:8192", per_token=True),
        # One GPU's share of a model split over heads (8 query heads on one
        # kv head): few sequences, long contexts.
        _decode("decode_shard_long", 16, 1, 8, 1, 64, "uniform:8192:32768"),
        # The speculative batch on 1024-token pages, work list planned once.
        _decode("decode_mtp_p1024", 256, 4, 64, 4, 1024, "uniform:4096:8192", per_token=True),
        # The serving step of a model with 64-wide heads.
        _decode("decode_d64", 64, 1, 32, 8, 16, "fixed:4096", head=64),
        # Prompt processing: four prompts of 4096 tokens into the fp8 cache.
        {"name": "rope_prefill", "family": "rope", "seqs": 4, "seq_tokens": 4096, "heads": 32, "kv_heads": 8,
         "head": 128, "page": 16, "cache": "fp8", "layout": "trans", "lengths": 7},
        # Query and KV rows of a prefill chunk, fp8 out with a scale per 128.
        {"name": "qknr_prefill", "family": "qknr", "tokens": 8192, "heads": 16, "head": 512, "rope": 64,
         "quant": True, "group": 128, "scale": "fp32"},
        # MLA decode of a few short contexts, and of a full serving batch.
        {"name": "mla_small", "family": "mla", "batch": 4, "ctx": "fixed:2048", "lengths": 7},
        {"name": "mla_b128", "family": "mla", "batch": 128, "ctx": "fixed:8192", "lengths": 7},
    ]


# (query heads, kv heads): the shapes of the listed cases and shards of them.
_HEADS = ((8, 2), (32, 8), (64, 8), (64, 4), (8, 1), (16, 1))
# Attended (token, kv head) pairs of a drawn decode: at most those of the
# speculative batch.
_MOST_PAIRS = 256 * 6000 * 4
_MOST_MLA = 128 * 8192


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_ctx(rng, lo, hi, most_mean):
    top = _log_int(rng, lo, max(lo + 1, min(hi, int(2 * most_mean))))
    kind = rng.choice(("fixed", "uniform", "uniform", "lognormal"))
    if kind == "fixed":
        return "fixed:%d" % min(top, max(lo, int(most_mean)))
    if kind == "uniform":
        return "uniform:%d:%d" % (max(lo, int(top * rng.uniform(0.0, 0.8) * 0.5)), top)
    return "lognormal:%d:1.0:%d:%d" % (max(lo, min(top, int(most_mean)) // 4), lo, max(lo + 1, top))


def draw(rng):
    family = rng.choice(("decode",) * 6 + ("layer", "rope", "qknr", "mla", "mla"))
    lengths = rng.randrange(1, 1 << 30)
    if family == "decode":
        heads, kv_heads = rng.choice(_HEADS)
        ql = rng.choice((1, 1, 1, 2, 3, 4))
        batch = _log_int(rng, 1, 256)
        page = rng.choice((16, 16, 64, 1024))
        head = rng.choice((128,) * 6 + (64, 256))
        ctx = _draw_ctx(rng, 16, 32768, min(32768, _MOST_PAIRS * 128 // head // (batch * kv_heads)))
        window = rng.choice((0, 0, 0, _log_int(rng, 128, 8192))) if page != 1024 else 0
        return _decode(None, batch, ql, heads, kv_heads, page, ctx, head=head, per_token=rng.random() < 0.5,
                       window=window, dtype=rng.choice(("bf16", "bf16", "bf16", "f16")), lengths=lengths)
    if family == "layer":
        heads, kv_heads = rng.choice(_HEADS)
        batch = _log_int(rng, 1, 64)
        return {"family": "layer", "batch": batch, "heads": heads, "kv_heads": kv_heads, "page": rng.choice((16, 64)),
                "ctx": _draw_ctx(rng, 1, MAX_POS, MAX_POS), "lengths": lengths}
    if family == "rope":
        heads, kv_heads = rng.choice(_HEADS)
        decode = rng.random() < 0.4
        tokens = _log_int(rng, 1, 512) if decode else _log_int(rng, 16, 16384)
        seqs = tokens if decode else rng.choice((1, 1, 2, 4))
        return {"family": "rope", "seqs": seqs, "seq_tokens": 1 if decode else min(MAX_POS, max(1, tokens // seqs)),
                "heads": heads, "kv_heads": kv_heads, "head": rng.choice((128, 128, 128, 64, 256)),
                "page": rng.choice((16, 16, 64)), "cache": rng.choice(("fp8", "fp8", "bf16")),
                "layout": rng.choice(("trans", "trans", "atom", "flash")), "lengths": lengths}
    if family == "qknr":
        quant = rng.random() < 0.75
        return {"family": "qknr", "tokens": _log_int(rng, 1, 8192), "heads": rng.choice((8, 16, 16)),
                "head": 512, "rope": 64, "quant": quant, "group": rng.choice((64, 128, 128)) if quant else 512,
                "scale": rng.choice(("fp32", "fp32", "e8m0")) if quant else "fp32"}
    batch = _log_int(rng, 1, 128)
    return {"family": "mla", "batch": batch, "ctx": _draw_ctx(rng, 16, 16384, min(16384, _MOST_MLA // batch)),
            "lengths": lengths}


def context_lengths(case):
    """Context length of every sequence: the case's own."""
    rng = np.random.default_rng(case["lengths"])
    kind, *p = case["ctx"].split(":")
    batch = case["batch"]
    if kind == "fixed":
        got = np.full(batch, int(p[0]))
    elif kind == "uniform":
        got = rng.integers(int(p[0]), int(p[1]) + 1, size=batch)
    else:
        x = np.exp(rng.normal(math.log(float(p[0])), float(p[1]), size=batch))
        got = np.clip(np.round(x), int(p[2]), int(p[3]))
    return [max(int(v), case.get("ql", 1)) for v in got]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rows_to_keys(q, page):  # [NB, H, bs, D] -> [NB, H, D/16, bs, 16]
    nb, h, _, d = q.shape
    return q.view(torch.uint8).reshape(nb, h, page, d // 16, 16).permute(0, 1, 3, 2, 4).contiguous().view(FP8)


def _rows_to_values(q, page):  # [NB, H, bs, D] -> [NB, H, bs/16, D, 16]
    nb, h, _, d = q.shape
    return q.view(torch.uint8).reshape(nb, h, page // 16, 16, d).permute(0, 1, 2, 4, 3).contiguous().view(FP8)


def _quantised(gen, shape, per_token):
    x = torch.randn(shape, generator=gen, device="cuda")
    amax = x.abs().amax(-1, keepdim=True) if per_token else x.abs().amax().reshape(1)
    scale = (amax / FP8_MAX).contiguous()
    return (x / scale).to(FP8), scale


def _pages(ctx, page, seed):
    """Block table and flat page list of sequences dealt randomly permuted
    pages, and the pool's size."""
    counts = [-(-c // page) for c in ctx]
    perm = np.random.default_rng(seed).permutation(sum(counts)).astype(np.int32)
    table = np.zeros((len(ctx), max(counts)), dtype=np.int32)
    at = 0
    for b, n in enumerate(counts):
        table[b, :n] = perm[at:at + n]
        at += n
    indptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    return table, perm, indptr, at


def _prepare_decode(case, seed):
    gen = _gen(seed)
    ctx = context_lengths(case)
    b, ql, hq, hkv, page, d = (case[k] for k in ("batch", "ql", "heads", "kv_heads", "page", "head"))
    table, flat, indptr, nb = _pages(ctx, page, seed)
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    query = torch.randn(b * ql, hq, d, generator=gen, device="cuda").to(dtype)
    k, ks = _quantised(gen, (nb, hkv, page, d), case["per_token"])
    key_cache = _rows_to_keys(k, page)
    del k
    v, vs = _quantised(gen, (nb, hkv, page, d), case["per_token"])
    value_cache = _rows_to_values(v, page)
    del v
    s = {"case": case, "query": query, "out": torch.empty_like(query), "keys": key_cache, "values": value_cache,
         "key_scale": ks, "value_scale": vs, "scale": 1.0 / math.sqrt(d),
         "lens": torch.tensor(ctx, dtype=torch.int32, device="cuda"), "table": None, "flat": None, "indptr": None,
         "more": {}}
    if page in (16, 64) or case["window"]:
        s["table"] = torch.from_numpy(table).cuda()
        # the split count a caller asks for, and, for windows, the partial
        # buffers that it keeps
        if case["window"]:
            p = get_recommended_splits(b, hkv, sliding_window=case["window"], query_length=ql)
            part = (b, hkv, p, ql * (hq // hkv))
            s["more"] = {"exp_sums": torch.empty(part, device="cuda"), "max_logits": torch.empty(part, device="cuda"),
                         "temporary_output": torch.empty(part + (d,), device="cuda", dtype=torch.bfloat16)}
        else:
            p = get_recommended_splits(b, hkv, split_kv_blocks=max(1, 256 // page))
        s["more"]["max_context_partition_num"] = p
    else:
        s["flat"], s["indptr"] = torch.from_numpy(flat).cuda(), torch.from_numpy(indptr).cuda()
        s["more"] = {"metadata": get_pa_metadata(query, key_cache, s["lens"], s["indptr"], hq, hkv)}
    return s


def _run_decode(s):
    pa_decode_ps_launch(s["out"], s["query"], s["keys"], s["values"], s["lens"], s["flat"], s["indptr"], s["scale"],
                        s["key_scale"], s["value_scale"], sliding_window=s["case"]["window"], block_tables=s["table"],
                        **s["more"])
    return {"out": s["out"]}


def _tables(d, dtype):
    inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.float64) / d))
    ang = torch.arange(MAX_POS, dtype=torch.float64)[:, None] * inv[None, :]
    return torch.cos(ang).to(dtype).cuda(), torch.sin(ang).to(dtype).cuda()


def _prepare_layer(case, seed):
    gen = _gen(seed)
    ctx = context_lengths(case)
    b, hq, hkv, page, d = case["batch"], case["heads"], case["kv_heads"], case["page"], 128
    table, _, _, nb = _pages(ctx, page, seed)
    bf16 = torch.bfloat16
    q = torch.randn(b, hq, d, generator=gen, device="cuda").to(bf16)
    k = torch.randn(b, hkv, d, generator=gen, device="cuda").to(bf16)
    v = torch.randn(b, hkv, d, generator=gen, device="cuda").to(bf16)
    one = torch.tensor([6.0 / FP8_MAX], dtype=torch.float32, device="cuda")
    rows = [(torch.randn(nb, hkv, page, d, generator=gen, device="cuda") / one).clamp(-FP8_MAX, FP8_MAX).to(FP8)
            for _ in range(2)]
    pos = np.array([c - 1 for c in ctx])
    slots = table[np.arange(b), pos // page].astype(np.int64) * page + pos % page
    cos, sin = _tables(d, bf16)
    return {"case": case, "q": q, "k": k, "v": v, "cos": cos, "sin": sin,
            "positions": torch.from_numpy(pos.astype(np.int32)).cuda(),
            "slots": torch.from_numpy(slots.astype(np.int32)).cuda(),
            "keys": _rows_to_keys(rows[0], page), "values": _rows_to_values(rows[1], page),
            "key_scale": one, "value_scale": one.clone(), "scale": 1.0 / math.sqrt(d),
            "lens": torch.tensor(ctx, dtype=torch.int32, device="cuda"), "table": torch.from_numpy(table).cuda(),
            "q_out": torch.empty_like(q), "k_out": torch.empty_like(k), "out": torch.empty_like(q),
            "splits": get_recommended_splits(b, hkv, split_kv_blocks=max(1, 256 // page)),
            "write": build_fused_rope_cache_module(head_dim=d, num_q_heads=hq, num_kv_heads=hkv, block_size=page,
                                                   flash_layout=False, dtype_str="bf16", apply_scale=True)}


def _run_layer(s):
    s["write"](s["q"], s["k"], s["v"], s["positions"], s["cos"], s["sin"], s["slots"], s["keys"], s["values"],
               s["q_out"], s["k_out"], s["q"].shape[0], s["key_scale"], s["value_scale"])
    pa_decode_ps_launch(s["out"], s["q_out"], s["keys"], s["values"], s["lens"], None, None, s["scale"],
                        s["key_scale"], s["value_scale"], block_tables=s["table"],
                        max_context_partition_num=s["splits"])
    return {"out": s["out"], "q": s["q_out"], "k": s["k_out"], "keys": s["keys"], "values": s["values"]}


def _prepare_rope(case, seed):
    gen = _gen(seed)
    seqs, n, hq, hkv, d, page = (case[k] for k in ("seqs", "seq_tokens", "heads", "kv_heads", "head", "page"))
    t = seqs * n
    bf16 = torch.bfloat16
    q = torch.randn(t, hq, d, generator=gen, device="cuda").to(bf16)
    k = torch.randn(t, hkv, d, generator=gen, device="cuda").to(bf16)
    v = torch.randn(t, hkv, d, generator=gen, device="cuda").to(bf16)
    cos, sin = _tables(d, bf16)
    rng = np.random.default_rng(seed)
    per = -(-n // page)
    nb = seqs * per + 64
    table = rng.permutation(nb)[:seqs * per].reshape(seqs, per)
    tok = np.arange(n)
    if n == 1:  # decode: the next token of contexts that already fill part of a page
        pos = np.random.default_rng(case["lengths"]).integers(1, MAX_POS, size=seqs)
        slots = table[:, 0] * page + pos % page
    else:
        pos = np.tile(tok, seqs)
        slots = (table[:, tok // page] * page + tok % page).reshape(-1)
    fp8 = case["cache"] == "fp8"
    shapes = {"trans": ((nb, hkv, d // 16, page, 16), (nb, hkv, page // 16, d, 16)),
              "atom": ((nb, hkv, d // 16, page, 16), (nb, hkv, d, page)),
              "flash": ((nb, page, hkv, d), (nb, page, hkv, d))}[case["layout"]]
    keys, values = (torch.zeros(x, dtype=torch.uint8 if fp8 else bf16, device="cuda") for x in shapes)
    return {"case": case, "q": q, "k": k, "v": v, "cos": cos, "sin": sin,
            "positions": torch.from_numpy(pos.astype(np.int32)).cuda(),
            "slots": torch.from_numpy(slots.astype(np.int32)).cuda(),
            "keys": keys.view(FP8) if fp8 else keys, "values": values.view(FP8) if fp8 else values,
            "key_scale": torch.tensor([8.0 / FP8_MAX], device="cuda"),
            "value_scale": torch.tensor([6.0 / FP8_MAX], device="cuda"),
            "q_out": torch.empty_like(q), "k_out": torch.empty_like(k),
            "write": build_fused_rope_cache_module(head_dim=d, num_q_heads=hq, num_kv_heads=hkv, block_size=page,
                                                   flash_layout=case["layout"] == "flash", dtype_str="bf16",
                                                   apply_scale=fp8)}


def _run_rope(s):
    s["write"](s["q"], s["k"], s["v"], s["positions"], s["cos"], s["sin"], s["slots"], s["keys"], s["values"],
               s["q_out"], s["k_out"], s["q"].shape[0], s["key_scale"], s["value_scale"])
    return {"q": s["q_out"], "k": s["k_out"], "keys": s["keys"], "values": s["values"]}


def _prepare_qknr(case, seed):
    gen = _gen(seed)
    t, h, d, rd = case["tokens"], case["heads"], case["head"], case["rope"]
    cos, sin = _tables(rd, torch.bfloat16)
    bf16 = torch.bfloat16
    return {"case": case, "q": torch.randn(t, h * d, generator=gen, device="cuda").to(bf16),
            "kv": torch.randn(t, d, generator=gen, device="cuda").to(bf16),
            "weight": (1.0 + 0.1 * torch.randn(d, generator=gen, device="cuda")).to(bf16), "cos": cos, "sin": sin,
            "positions": torch.randint(0, MAX_POS, (t,), generator=gen, device="cuda")}


def _run_qknr(s):
    c = s["case"]
    q, kv, qs, kvs = flydsl_qk_norm_rope_quant(
        s["q"], s["kv"], s["weight"], s["cos"], s["sin"], s["positions"], num_q_heads=c["heads"],
        head_dim=c["head"], rope_head_dim=c["rope"], quant=c["quant"],
        quant_group_size=c["group"] if c["quant"] else None, scale_dtype=c["scale"])
    return {"q": q, "kv": kv, "q_scale": qs, "kv_scale": kvs}


def _prepare_mla(case, seed):
    gen = _gen(seed)
    ctx = context_lengths(case)
    b, total = case["batch"], sum(ctx)
    q = torch.randn(b, 128, 576, generator=gen, device="cuda").to(FP8)
    kv = torch.randn(total, 1, 1, 576, generator=gen, device="cuda").to(FP8)
    indices = torch.randperm(total, generator=gen, device="cuda").to(torch.int32)
    kv_indptr = torch.tensor([0] + list(np.cumsum(ctx)), dtype=torch.int32)
    qo_indptr = torch.arange(b + 1, dtype=torch.int32)
    last = torch.ones(b, dtype=torch.int32)
    meta = [torch.empty(n, dtype=t, device="cuda") for n, t in get_mla_metadata_info_v1(b, 1, 128, FP8, FP8)]
    get_mla_metadata_v1(qo_indptr, kv_indptr, last, 128, 1, True, meta[0], meta[2], meta[1], meta[3], meta[4],
                        meta[5], kv_granularity=16, max_seqlen_qo=1, uni_seqlen_qo=1)
    parts = max(1, int(meta[0][2]))
    return {"case": case, "q": q, "kv": kv, "indices": indices, "kv_indptr": kv_indptr, "meta": meta,
            "scale": 1.0 / math.sqrt(576), "out": torch.empty(b, 128, 512, device="cuda", dtype=torch.bfloat16),
            "split": torch.empty(parts, 1, 128, 512, device="cuda"), "lse": torch.empty(parts, 1, 128, 1, device="cuda")}


def _run_mla(s):
    _, indptr, info, reduce_indptr, final_map, partial_map = s["meta"]
    flydsl_mla_fwd_decode(s["q"], s["kv"], s["indices"], indptr, info, s["out"], s["split"], s["lse"], s["scale"])
    mla_reduce_v1(s["split"], s["lse"], reduce_indptr, final_map, partial_map, 1, s["out"])
    return {"out": s["out"]}


_PREPARE = {"decode": _prepare_decode, "layer": _prepare_layer, "rope": _prepare_rope, "qknr": _prepare_qknr,
            "mla": _prepare_mla}
_RUN = {"decode": _run_decode, "layer": _run_layer, "rope": _run_rope, "qknr": _run_qknr, "mla": _run_mla}


def prepare(case, seed):
    return _PREPARE[case["family"]](case, seed)


def run(state):
    return _RUN[state["case"]["family"]](state)


# ---------------------------------------------------------------------------
# Work and precision
# ---------------------------------------------------------------------------


def _attended(case, ctx):
    """(distinct keys read, (query token, key) pairs) over the batch."""
    ql, window = case.get("ql", 1), case.get("window", 0)
    keys = pairs = 0
    for c in ctx:
        keys += min(c, ql + window) if window else c
        for i in range(ql):
            n = c - ql + 1 + i
            pairs += min(n, window + 1) if window else n
    return keys, pairs


def work(case):
    f = case["family"]
    if f in ("decode", "layer"):
        ctx = context_lengths(case)
        keys, pairs = _attended(case, ctx)
        d, hkv, hq = case.get("head", 128), case["kv_heads"], case["heads"]
        rows = case["batch"] * case.get("ql", 1) * hq
        per_key = hkv * (2 * d + (8 if case.get("per_token") else 0))
        got = {"bytes": keys * per_key + 2 * rows * d * 2, "flops": pairs * hq * d * 4}
        if f == "layer":
            got["bytes"] += _rope_bytes(case["batch"], hq, hkv, d, 1)
            got["flops"] += case["batch"] * (hq + hkv) * d * 3
        return got
    if f == "rope":
        t, el = case["seqs"] * case["seq_tokens"], 1 if case["cache"] == "fp8" else 2
        return {"bytes": _rope_bytes(t, case["heads"], case["kv_heads"], case["head"], el),
                "flops": t * (case["heads"] + case["kv_heads"]) * case["head"] * 3}
    if f == "qknr":
        d, rows = case["head"], case["heads"] + 1
        out = d + d // case["group"] * (4 if case["scale"] == "fp32" else 1) if case["quant"] else 2 * d
        return {"bytes": case["tokens"] * (rows * (2 * d + out) + 8 + 2 * case["rope"]) + 2 * d,
                "flops": case["tokens"] * rows * d * 6}
    ctx = context_lengths(case)
    return {"bytes": sum(ctx) * 580 + case["batch"] * 128 * (576 + 1024),
            "flops": sum(ctx) * 128 * (576 + 512) * 2}


def _rope_bytes(tokens, hq, hkv, d, cache_el):
    return tokens * ((hq + 2 * hkv) * d * 2 + 2 * d + 8 + (hq + hkv) * d * 2 + 2 * hkv * d * cache_el)


def tolerance(case):
    f = case["family"]
    if f == "decode":
        # 16-bit outputs of fp8 products carried in two terms each
        return {"rel": 1e-2, "max": 0.1}
    if f == "layer":
        return {"rel": 1e-2, "max": 0.1}
    if f == "rope":
        # the rotation's roundings are part of the format: every product and
        # sum is rounded to 16 bits, and the cache bytes are quantised from that
        return "exact"
    if f == "qknr":
        # one 16-bit or fp8 step where a sum's order moves a value across a tie
        # (a group at a tie of its e8m0 exponent moves by a factor of two)
        if case["quant"] and case["scale"] == "e8m0":
            return {"rel": 5e-3, "max": 1.0 - 1e-9, "differ": 1e-3}
        return {"rel": 5e-3, "max": 0.15}
    # the probabilities are single fp8 terms (relative error up to 2^-4 each)
    return {"rel": 3e-2, "max": 0.3}


def _exact_attention(query, keys, values, key_scale, value_scale, table, ctx, scale, ql, window, page):
    """Attention over a paged cache in 64 bits: [B*ql, Hq, D]."""
    hq, d = query.shape[1:]
    hkv = keys.shape[1]
    gqa = hq // hkv
    out = torch.zeros(query.shape, dtype=torch.float64, device=query.device)
    for b, n in enumerate(ctx):
        lo = max(0, n - ql - window) // page * page if window else 0
        pages = table[b, lo // page:-(-n // page)].long()
        k = keys[pages].to(torch.float64).permute(1, 0, 3, 2, 4).reshape(hkv, -1, d)
        v = values[pages].to(torch.float64).permute(1, 0, 2, 4, 3).reshape(hkv, -1, d)
        if key_scale.dim() > 1:
            k = k * key_scale[pages].to(torch.float64).permute(1, 0, 2, 3).reshape(hkv, -1, 1)
            v = v * value_scale[pages].to(torch.float64).permute(1, 0, 2, 3).reshape(hkv, -1, 1)
        else:
            k, v = k * key_scale.to(torch.float64), v * value_scale.to(torch.float64)
        k, v = k[:, :n - lo].contiguous(), v[:, :n - lo].contiguous()
        q = query[b * ql:(b + 1) * ql].to(torch.float64).reshape(ql, hkv, gqa, d).permute(1, 0, 2, 3)
        x = torch.matmul(q.reshape(hkv, ql * gqa, d), k.transpose(1, 2).contiguous()) * scale
        at = torch.arange(lo, n, device=x.device)
        row = torch.arange(n - ql, n, device=x.device).repeat_interleave(gqa)
        hide = at[None, :] > row[:, None]
        if window:
            hide |= at[None, :] < row[:, None] - window
        x = x.masked_fill(hide[None], -math.inf)
        o = torch.matmul(torch.softmax(x, -1), v)
        out[b * ql:(b + 1) * ql] = o.reshape(hkv, ql, gqa, d).permute(1, 0, 2, 3).reshape(ql, hq, d)
    return out


def _rotated(x, cos, sin):
    """NeoX rotation in 64 bits, and with every product and sum rounded to 16."""
    h = x.shape[-1] // 2
    c, s = cos[:, None, :], sin[:, None, :]
    a, b = x[..., :h], x[..., h:]
    got = torch.cat([a * c - b * s, b * c + a * s], -1)  # rounded by torch's 16-bit arithmetic
    a, b, c, s = (t.to(torch.float64) for t in (a, b, c, s))
    return torch.cat([a * c - b * s, b * c + a * s], -1), got


def _to_fp8(x, scale):
    """Value bytes as the writer stores them: x times the float32 reciprocal."""
    return (x.to(torch.float32) * (1.0 / scale)).clamp(-FP8_MAX, FP8_MAX).to(FP8)


def exact(case, seed):
    s = prepare(case, seed)
    f = case["family"]
    if f == "decode":
        ctx = context_lengths(case)
        table = torch.from_numpy(_pages(ctx, case["page"], seed)[0]).cuda()
        return {"out": _exact_attention(s["query"], s["keys"], s["values"], s["key_scale"], s["value_scale"], table,
                                        ctx, s["scale"], case["ql"], case["window"], case["page"])}
    if f == "layer":
        ctx = context_lengths(case)
        pos, page = s["positions"].long(), case["page"]
        q, q16 = _rotated(s["q"], s["cos"][pos], s["sin"][pos])
        k, k16 = _rotated(s["k"], s["cos"][pos], s["sin"][pos])
        slots = s["slots"].long()
        nb, hkv = s["keys"].shape[:2]
        keys, values = s["keys"].view(torch.uint8).clone(), s["values"].view(torch.uint8).clone()
        k8, v8 = (_to_fp8(t, s["key_scale"]).view(torch.uint8) for t in (k16, s["v"]))
        at = slots % page
        keys[slots // page, :, :, at, :] = k8.reshape(-1, hkv, 8, 16)
        values[slots // page, :, at // 16, :, at % 16] = v8
        return {"out": _exact_attention(q16, keys.view(FP8), values.view(FP8), s["key_scale"], s["value_scale"],
                                        s["table"], ctx, s["scale"], 1, 0, page),
                "q": q, "k": k, "keys": None, "values": None}
    if f == "rope":
        pos = s["positions"].long()
        return {"q": _rotated(s["q"], s["cos"][pos], s["sin"][pos])[0],
                "k": _rotated(s["k"], s["cos"][pos], s["sin"][pos])[0], "keys": None, "values": None}
    if f == "qknr":
        return _exact_qknr(case, s)
    out = torch.empty(s["out"].shape, dtype=torch.float64, device="cuda")
    for b in range(case["batch"]):
        rows = s["kv"][s["indices"][s["kv_indptr"][b]:s["kv_indptr"][b + 1]].long()].reshape(-1, 576)
        rows = rows.to(torch.float64)
        x = torch.matmul(s["q"][b].to(torch.float64), rows.t().contiguous()) * s["scale"]
        out[b] = torch.matmul(torch.softmax(x, -1), rows[:, :512].contiguous())
    return {"out": out}


def _exact_qknr(case, s):
    t, h, d, rd = case["tokens"], case["heads"], case["head"], case["rope"]
    x = torch.cat([s["q"].view(t, h, d), s["kv"][:, None, :]], 1).to(torch.float64)
    rstd = torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
    x[:, h:] *= s["weight"].to(torch.float64)
    c, n = (tab[s["positions"]].to(torch.float64)[:, None, :] for tab in (s["cos"], s["sin"]))
    a, b = x[..., d - rd::2], x[..., d - rd + 1::2]
    y = x.clone()
    y[..., d - rd::2], y[..., d - rd + 1::2] = a * c - b * n, b * c + a * n
    if not case["quant"]:
        y = y * rstd
        return {"q": y[:, :h], "kv": y[:, h], "q_scale": None, "kv_scale": None}
    # one scale per group of the unrotated row: amax * sqrt(2) / 448, or the
    # e8m0 exponent byte of amax * sqrt(2) rounded to a power of two, less 7
    g = case["group"]
    amax = x.abs().reshape(t, h + 1, d // g, g).amax(-1)
    if case["scale"] == "e8m0":
        bits = (amax * rstd * math.sqrt(2.0)).to(torch.float32).view(torch.int32)
        byte = ((bits + 0x400000) >> 23) - 7
        factor, sc = rstd * torch.exp2((127 - byte).to(torch.float64)), None
    else:
        factor, sc = FP8_MAX / math.sqrt(2.0) / amax, amax * rstd * (math.sqrt(2.0) / FP8_MAX)
    y = (y.reshape(t, h + 1, d // g, g) * factor[..., None]).reshape(t, h + 1, d)
    return {"q": y[:, :h], "kv": y[:, h], "q_scale": None if sc is None else sc[:, :h],
            "kv_scale": None if sc is None else sc[:, h]}
