"""The work that a program has this package do, as measurable cases.

A serving engine calls the package once per layer and generated token: it
appends the token's key and value (or latent) rows to a paged cache and
attends over the pages of every sequence of the batch.  The cases are those
calls through the public entry points, from a handful of short sequences to
multi-gigabyte contexts, for the data types, head shapes and page sizes that
caches are kept in.

A case is a dict of plain values.  Lengths follow from the case alone (so
that its work is known); the seed gives the order of the sequences, the page
order and every tensor.
"""
from __future__ import annotations

import math
import random

import torch

import attention_amd

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}

# DeepSeek-V3 attention dimensions: no-rope query, latent, rope and value.
DN, DC, DR, DV = 128, 512, 64, 128


def _gqa(name, op, dtype, batch, q_heads, kv_heads, head_dim, block_size, lo, hi, *, k_scale=1.0, slack=1.0,
         splits=0):
    """``slack``: block-table width over the longest sequence's pages (an
    engine sizes the table for its longest allowed context).  ``k_scale``
    widens the scores: trained models attend to few tokens, unlike N(0,1)
    keys."""
    case = dict(op=op, dtype=dtype, batch=batch, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                block_size=block_size, len_lo=lo, len_hi=hi, k_scale=k_scale, slack=slack, splits=splits)
    return dict(case, name=name) if name else case


def _mla(name, op, dtype, batch, q_len, heads, block_size, lo, hi, *, selected=0):
    """``q_len`` queries per sequence (more than one: speculated tokens);
    ``selected``: tokens listed per query, 0 for all of the context."""
    case = dict(op=op, dtype=dtype, batch=batch, q_len=q_len, heads=heads, block_size=block_size, len_lo=lo,
                len_hi=hi, selected=selected)
    return dict(case, name=name) if name else case


def listed():
    return [
        # A few short prompts on a small model: launches and latency.
        _gqa("gqa-small", "gqa", "fp16", 4, 8, 2, 64, 16, 17, 512),
        # The headline shape: a mid-size batch of chat contexts (Qwen3-8B).
        _gqa("gqa-serve", "gqa", "bf16", 32, 32, 8, 128, 16, 512, 4096),
        # A whole decode step of a layer, append and attend, high batch of
        # short contexts.
        _gqa("gqa-step", "step", "fp16", 128, 40, 8, 128, 32, 128, 1024, slack=2.0),
        # Long documents: the largest calls.
        _gqa("gqa-long", "gqa", "bf16", 8, 64, 8, 128, 16, 32768, 131072, k_scale=3.0),
        # fp32 caches (the reference's sweep runs them): numerics work and
        # evaluation.
        _gqa("gqa-fp32", "gqa", "fp32", 16, 32, 8, 128, 16, 64, 1024),
        # A head_dim that is no power of two (Phi-2: 80), every head its own
        # keys.
        _gqa("gqa-d80", "gqa", "fp16", 16, 32, 32, 80, 16, 256, 2048),
        # Small pages: engines that share prefixes finely keep 1 to 8 tokens
        # per page.
        _gqa("gqa-page8", "gqa", "bf16", 24, 32, 8, 128, 8, 128, 3000, k_scale=2.0),
        # A caller that plans its own splits and keeps the workspace.
        _gqa("gqa-split", "split", "bf16", 4, 32, 8, 128, 16, 2048, 4096, splits=16),
        # MLA, the 16-head share of a tensor-parallel rank.
        _mla("mla-tp16", "mla", "bf16", 128, 1, 16, 64, 1024, 4096),
        # MLA, all 128 heads on one GPU: the matrix-core end.
        _mla("mla-h128", "mla", "bf16", 32, 1, 128, 64, 1024, 4096),
        # MLA over selected tokens of long contexts (sparse attention).
        _mla("mla-sparse", "mla", "bf16", 16, 1, 128, 64, 4096, 16384, selected=2048),
        # MLA decode step with one speculated token: latent write, then two
        # queries per sequence.
        _mla("mla-step2", "mla-step", "fp16", 48, 2, 32, 64, 512, 4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.68:
        op = rng.choice(["gqa", "gqa", "gqa", "gqa", "step", "split"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"])
        head_dim = rng.choice([64, 128, 128, 128, 256, 96, 80, 72, 112, 160, 192])
        block_size = rng.choice([16, 16, 16, 32, 64, 128, 8, 1, 12])
        kv_heads, group = rng.choice([(8, 4), (8, 4), (8, 5), (8, 8), (4, 7), (4, 8), (2, 4), (1, 8), (1, 32),
                                      (32, 1), (12, 1), (16, 2), (3, 3)])
        hi = _log_int(rng, 32, 65536)
        lo = rng.choice([1, max(1, hi // 8), max(1, hi // 2), hi])
        token = 2 * kv_heads * head_dim * BYTES[dtype]
        # What the tuned shapes read in a call of the largest listed case;
        # the other shapes take several times as long per byte.
        tuned = head_dim in (64, 128, 256) and block_size % 16 == 0 and dtype != "fp32"
        room = (1_200_000_000 if tuned else 150_000_000) / token
        hi = int(min(hi, room))
        lo = min(lo, hi)
        batch = _log_int(rng, 1, max(1, min(256, int(room / ((lo + hi) / 2)))))
        return _gqa("", op, dtype, batch, group * kv_heads, kv_heads, head_dim, block_size, lo, hi,
                    k_scale=rng.choice([1.0, 2.0, 3.0]), slack=rng.choice([1.0, 1.0, 2.0]),
                    splits=rng.choice([2, 4, 8, 16, 64]) if op == "split" else 0)
    op = rng.choice(["mla", "mla", "mla", "mla-step"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    q_len = rng.choice([1, 1, 1, 2, 3, 4])
    heads = rng.choice([8, 16, 16, 20, 32, 64, 128, 128])
    selected = rng.choice([0, 0, 0, 256, 2048])
    block_size = rng.choice([64, 64, 32, 16, 128, 1])
    hi = _log_int(rng, 64, 32768)
    lo = rng.choice([max(1, hi // 8), max(1, hi // 2), hi])
    per_seq = q_len * max(16, heads) * (min(selected, hi) if selected else (lo + hi) / 2)
    room = 128 * 1200 * 16 if (selected or block_size == 1) else 128 * 2560 * 16
    batch = _log_int(rng, 1, max(1, min(256, int(room / per_seq))))
    return _mla("", op, dtype, batch, q_len, heads, block_size, lo, hi, selected=selected)


# ----------------------------------------------------------------------------
# Inputs
# ----------------------------------------------------------------------------


def _lengths(case):
    """The batch's context lengths (queries included), from the case alone."""
    lo, hi = max(case["len_lo"], case.get("q_len", 1)), case["len_hi"]
    rng = random.Random(f"{case['batch']}-{lo}-{hi}-{case['block_size']}")
    return [rng.randint(lo, max(lo, hi)) for _ in range(case["batch"])]


def _paged(case, seed):
    """(lengths, block table, pages of the pool, generator): sequences in the
    seed's order, their pages scattered over a pool of exactly those pages."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lens = _lengths(case)
    random.Random(seed).shuffle(lens)
    page = case["block_size"]
    used = [-(-n // page) for n in lens]
    width = max(1, math.ceil(max(used) * case.get("slack", 1.0)))
    order = torch.randperm(sum(used), generator=gen, device="cuda", dtype=torch.int32)
    counts = torch.tensor(used, device="cuda")
    col = torch.arange(width, device="cuda")[None, :]
    first = (counts.cumsum(0) - counts)[:, None]
    taken = col < counts[:, None]
    table = torch.where(taken, order[(first + col).clamp(max=sum(used) - 1)], -1).to(torch.int32).contiguous()
    return lens, table, sum(used), gen


def _randn(gen, *shape, dtype, scale=1.0):
    x = torch.randn(*shape, generator=gen, device="cuda", dtype=dtype)
    return x.mul_(scale) if scale != 1.0 else x


def prepare(case, seed):
    dtype = DTYPES[case["dtype"]]
    lens, table, pages, gen = _paged(case, seed)
    state = {"op": case["op"], "table": table, "lens": torch.tensor(lens, dtype=torch.int32, device="cuda")}
    b, page = case["batch"], case["block_size"]
    if "head_dim" in case:
        hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
        state["q"] = _randn(gen, b, hq, d, dtype=dtype)
        state["k"] = _randn(gen, pages, page, hkv, d, dtype=dtype, scale=case["k_scale"])
        state["v"] = _randn(gen, pages, page, hkv, d, dtype=dtype)
        if case["op"] == "step":
            state["key"] = _randn(gen, b, hkv, d, dtype=dtype, scale=case["k_scale"])
            state["value"] = _randn(gen, b, hkv, d, dtype=dtype)
            state["last"] = state["lens"] - 1
        if case["op"] == "split":
            state["splits"] = case["splits"]
            state["workspace"] = torch.empty(b, hq, case["splits"], d + 2, dtype=torch.float32, device="cuda")
        return state
    t, h = case["q_len"], case["heads"]
    state["q_nope"] = _randn(gen, b, t, h, DN, dtype=dtype)
    state["q_rope"] = _randn(gen, b, t, h, DR, dtype=dtype)
    state["cache"] = _randn(gen, pages, page, DC + DR, dtype=dtype)
    state["w_uk"] = _randn(gen, h, DN, DC, dtype=dtype, scale=DN ** -0.5)
    state["w_uv"] = _randn(gen, h, DV, DC, dtype=dtype, scale=DC ** -0.5)
    at = state["lens"][:, None] - t + torch.arange(t, device="cuda", dtype=torch.int32)[None, :]
    state["positions"] = at.to(torch.int32).contiguous()
    if case["op"] == "mla-step":
        state["latent"] = _randn(gen, b * t, DC, dtype=dtype)
        state["rope_key"] = _randn(gen, b * t, DR, dtype=dtype)
        where = torch.gather(table.long(), 1, (at // page).long())
        state["slots"] = (where * page + at % page).reshape(-1).contiguous()
    if case["selected"]:
        # Distinct visible tokens in ascending blocks of random ones, as a
        # top-k over index scores leaves them; short contexts are padded -1.
        k = case["selected"]
        draw = torch.rand(b, t, max(int(max(lens)), k), generator=gen, device="cuda")
        hidden = torch.arange(draw.shape[2], device="cuda")[None, None, :] > at[:, :, None]
        score, chosen = draw.masked_fill_(hidden, -1.0).topk(k, dim=2)
        state["indices"] = torch.where(score >= 0, chosen, -1).to(torch.int32).contiguous()
    return state


# ----------------------------------------------------------------------------
# One pass
# ----------------------------------------------------------------------------


def run(state):
    s, op = state, state["op"]
    if op == "gqa":
        return attention_amd.gqa_decode(s["q"], s["k"], s["v"], s["table"], s["lens"])
    if op == "step":
        attention_amd.kv_append(s["key"], s["value"], s["k"], s["v"], s["table"], s["last"])
        out = attention_amd.gqa_decode(s["q"], s["k"], s["v"], s["table"], s["lens"])
        return {"out": out, "k": s["k"], "v": s["v"]}
    if op == "split":
        return attention_amd.gqa_decode_split(s["q"], s["k"], s["v"], s["table"], s["lens"], splits=s["splits"],
                                              workspace=s["workspace"])
    if op == "mla-step":
        attention_amd.latent_kv_write(s["latent"], s["rope_key"], s["cache"], s["slots"])
    args = (s["q_nope"], s["q_rope"], s["cache"], s["table"], s["lens"], s["positions"], s["w_uk"], s["w_uv"])
    if "indices" in s:
        out = attention_amd.sparse_mla(*args, s["indices"])
    else:
        out = attention_amd.mla_decode(*args)
    return {"out": out, "cache": s["cache"]} if op == "mla-step" else out


def work(case):
    lens, e, b = _lengths(case), BYTES[case["dtype"]], case["batch"]
    pages = sum(-(-n // case["block_size"]) for n in lens)
    meta = 4 * b + 4 * pages
    if "head_dim" in case:
        row = case["kv_heads"] * case["head_dim"] * e
        qo = 2 * b * case["q_heads"] * case["head_dim"] * e
        append = 4 * b * row if case["op"] == "step" else 0
        return {"bytes": sum(lens) * 2 * row + qo + meta + append,
                "flops": 4 * case["q_heads"] * case["head_dim"] * sum(lens)}
    t, h = case["q_len"], case["heads"]
    seen = [[min(n - t + i + 1, case["selected"] or n) for i in range(t)] for n in lens]
    # All of a context is read once for its queries; listed rows once each.
    rows = sum(sum(s) if case["selected"] else n for n, s in zip(lens, seen))
    pairs = sum(sum(s) for s in seen)
    weights = h * (DN + DV) * DC
    append = 2 * b * t * (DC + DR) * e if case["op"] == "mla-step" else 0
    index = 4 * b * t * case["selected"]
    return {"bytes": (rows * (DC + DR) + b * t * h * (DN + DR + DV) + weights) * e + meta + 4 * b * t + append + index,
            "flops": 2 * h * pairs * (2 * DC + DR) + 2 * b * t * weights}


def tolerance(case):
    """About four times the distance to 64 bits of one pass: the output's own
    rounding (GQA), and for MLA the rounded absorbed query and latent output
    as well, which the operator's definition has."""
    if "head_dim" in case:
        return {"rel": {"bf16": 7e-3, "fp16": 1e-3, "fp32": 2.5e-6}[case["dtype"]]}
    return {"rel": {"bf16": 1.4e-2, "fp16": 2e-3}[case["dtype"]]}


# ----------------------------------------------------------------------------
# The same in 64 bits
# ----------------------------------------------------------------------------


def _softmax_sum(scores, values):
    """softmax(scores) @ values over the last axis of scores."""
    return torch.softmax(scores, -1) @ values


def exact(case, seed):
    s = prepare(case, seed)
    lens, table, page = s["lens"].tolist(), s["table"].long(), case["block_size"]
    if "head_dim" in case:
        if case["op"] == "step":
            rows = torch.gather(table, 1, (s["last"] // page).long()[:, None])[:, 0]
            s["k"][rows, (s["last"] % page).long()] = s["key"]
            s["v"][rows, (s["last"] % page).long()] = s["value"]
        hkv, d = case["kv_heads"], case["head_dim"]
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
        for i, n in enumerate(lens):
            ids = table[i, : -(-n // page)]
            k = s["k"][ids].reshape(-1, hkv, d)[:n]
            v = s["v"][ids].reshape(-1, hkv, d)[:n]
            for j in range(hkv):
                q = s["q"][i].view(hkv, -1, d)[j].double()
                out[i].view(hkv, -1, d)[j] = _softmax_sum(q @ k[:, j].double().t().contiguous() / math.sqrt(d),
                                                          v[:, j].double())
        return {"out": out, "k": None, "v": None} if case["op"] == "step" else out
    if case["op"] == "mla-step":
        flat = s["cache"].view(-1, DC + DR)
        flat[s["slots"], :DC] = s["latent"]
        flat[s["slots"], DC:] = s["rope_key"]
    b, t, h = case["batch"], case["q_len"], case["heads"]
    absorbed = torch.matmul(s["q_nope"].double().view(b * t, h, DN).transpose(0, 1).contiguous(), s["w_uk"].double())
    absorbed = absorbed.transpose(0, 1).reshape(b, t, h, DC)
    latent = torch.empty(b, t, h, DC, dtype=torch.float64, device="cuda")
    for i, n in enumerate(lens):
        context = s["cache"][table[i, : -(-n // page)]].reshape(-1, DC + DR)
        for u in range(t):
            rows = context[: n - t + u + 1]
            if case["selected"]:
                chosen = s["indices"][i, u]
                rows = rows[chosen[chosen >= 0].long()]
            rows = rows.double()
            query = torch.cat([absorbed[i, u], s["q_rope"][i, u].double()], -1)
            latent[i, u] = _softmax_sum(query @ rows.t().contiguous() / math.sqrt(DN + DR), rows[:, :DC])
    up = s["w_uv"].double().transpose(1, 2).contiguous()
    out = torch.matmul(latent.view(b * t, h, DC).transpose(0, 1).contiguous(), up)
    out = out.transpose(0, 1).reshape(b, t, h, DV).contiguous()
    return {"out": out, "cache": None} if case["op"] == "mla-step" else out
