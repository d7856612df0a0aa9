"""The framework's measured work: one dict of plain values per case, and the functions that
prepare, run, count and check it.

Kinds of cases (each runs the public operators of lightllm_amd.kv_cache, as an engine's step
calls them for one layer):

    decode         paged_decode: one new query token per sequence over its cached pages
    decode_append  paged_decode_append: the step's new K/V rows appended, then the decode
    prefill        paged_prefill: causal chunks on cached prefixes, several sequences at once
    first_prefill  scatter_prefill_kv_batched and first_prefill_attn_batched: new prompts
    rope_append    build_slots and rope_append: slot mapping, rotation, append of a step's rows
    gather         gather_kv: the pages of several sequences into contiguous rows

Pools are [pages, 16, kv heads, head_dim] with a quarter more pages than the batch needs, in a
random order, as an allocator that has run for a while hands them out.  q, k and v are N(0, 1),
so that scores have a standard deviation of one.
"""
from __future__ import annotations

import math
import random

import torch

PAGE = 16
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
DEVICE = "cuda"

# Head layouts (q heads, kv heads, head_dim) of the repository's configurations and tests.
LAYOUTS = [(14, 2, 64), (32, 8, 128), (32, 8, 128), (28, 4, 128), (12, 2, 128), (32, 32, 96), (16, 8, 256)]


def listed():
    return [
        # One user's chat turn: the smallest call, where launches and latency count.
        {"name": "decode_one_f32", "kind": "decode_append", "dtype": "f32", "hq": 14, "hkv": 2, "d": 64,
         "batch": 1, "lens": "fixed", "low": 512, "high": 512, "splits": 0},
        # A served batch of short and medium contexts in the reference's default type.
        {"name": "decode_b64_f32", "kind": "decode_append", "dtype": "f32", "hq": 14, "hkv": 2, "d": 64,
         "batch": 64, "lens": "uniform", "low": 129, "high": 2049, "splits": 0},
        # Few users with long documents; 1% of K entries are outliers.
        {"name": "decode_long_b16_f16", "kind": "decode", "dtype": "f16", "hq": 14, "hkv": 2, "d": 64,
         "batch": 16, "lens": "fixed", "low": 32768, "high": 32768, "splits": 0, "outliers": 0.01},
        # A full server: many sequences of very uneven lengths, grouped heads of 128.
        {"name": "decode_b256_f16", "kind": "decode_append", "dtype": "f16", "hq": 32, "hkv": 8, "d": 128,
         "batch": 256, "lens": "lognormal", "median": 1024, "low": 17, "high": 16385, "splits": 0},
        # Wide heads in bfloat16, an odd batch.
        {"name": "decode_b61_bf16_d256", "kind": "decode_append", "dtype": "bf16", "hq": 16, "hkv": 8, "d": 256,
         "batch": 61, "lens": "uniform", "low": 100, "high": 2100, "splits": 0},
        # Chunked prefill of eight requests, three of them on one shared prefix.
        {"name": "prefill_f16_d64", "kind": "prefill", "dtype": "f16", "hq": 14, "hkv": 2, "d": 64,
         "chunks": "512,512,512,512,512,512,512,512", "prefixes": "0,256,1024,4096,4096,4096,2048,512"},
        # Four long chunks on a system prompt of 2048 tokens.
        {"name": "prefill_f16_d128", "kind": "prefill", "dtype": "f16", "hq": 32, "hkv": 8, "d": 128,
         "chunks": "1024,1024,1024,1024", "prefixes": "2048,2048,2048,2048"},
        # A mixed queue of odd chunks: one new token to over a thousand, on odd prefixes.
        {"name": "prefill_bf16_ragged", "kind": "prefill", "dtype": "bf16", "hq": 32, "hkv": 8, "d": 128,
         "chunks": "1,37,129,700,1101,255,16", "prefixes": "901,0,2047,333,1200,64,3000"},
        # The eight requests in the reference's default type.
        {"name": "prefill_f32_d64", "kind": "prefill", "dtype": "f32", "hq": 14, "hkv": 2, "d": 64,
         "chunks": "512,512,512,512,512,512,512,512", "prefixes": "0,256,1024,4096,4096,4096,2048,512"},
        # Eight new prompts without a cached prefix.
        {"name": "first_prefill_f32_d64", "kind": "first_prefill", "dtype": "f32", "hq": 14, "hkv": 2, "d": 64,
         "chunks": "512,300,512,77,512,409,512,512"},
        # The rows of a mixed step: 256 decode tokens and four chunks of 1024.
        {"name": "rope_append_f16", "kind": "rope_append", "dtype": "f16", "hq": 32, "hkv": 8, "d": 128,
         "batch": 260, "tokens": 4352},
        # Cached contexts copied out of the pool.
        {"name": "gather_bf16", "kind": "gather", "dtype": "bf16", "hq": 32, "hkv": 8, "d": 128,
         "batch": 48, "lens": "uniform", "low": 100, "high": 3000},
    ]


# What a drawn case may cost at most (the largest listed cases' work).
_MAX_KV_BYTES = 1_300_000_000
_MAX_FLOPS = {"f32": 2e10, "f16": 1e11, "bf16": 1e11}


def _log_int(rng: random.Random, low: int, high: int) -> int:
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["decode", "decode_append", "decode_append", "prefill", "prefill", "prefill",
                       "first_prefill", "rope_append", "gather"])
    hq, hkv, d = rng.choice(LAYOUTS)
    c = {"kind": kind, "dtype": rng.choice(["f32", "f16", "bf16", "bf16"]), "hq": hq, "hkv": hkv, "d": d}
    row_bytes = 2 * hkv * d * DTYPES[c["dtype"]].itemsize
    if kind in ("decode", "decode_append", "gather"):
        c["batch"] = _log_int(rng, 1, 256)
        most = max(64, min(32768, int(_MAX_KV_BYTES / (2 if kind == "gather" else 1) / (row_bytes * c["batch"]))))
        high = _log_int(rng, 64, most)
        c.update(lens=rng.choice(["uniform", "uniform", "lognormal"]), low=max(1, high // rng.choice([2, 16])), high=high)
        if kind != "gather":
            c["splits"] = rng.choice([0, 0, 0, 0, 4, 16])
    elif kind in ("prefill", "first_prefill"):
        n = rng.randint(1, 9)
        chunks = [_log_int(rng, 1, 1500) for _ in range(n)]
        prefixes = [0] * n if kind == "first_prefill" else [rng.choice([0, _log_int(rng, 16, 4500)]) for _ in range(n)]
        while sum(_pairs(p, x) for p, x in zip(prefixes, chunks)) * 4 * d * hq > _MAX_FLOPS[c["dtype"]]:
            chunks = [max(1, x // 2) for x in chunks]
        c["chunks"] = ",".join(map(str, chunks))
        if kind == "prefill":
            c["prefixes"] = ",".join(map(str, prefixes))
    else:
        c["tokens"] = _log_int(rng, 1, 6000 if c["dtype"] != "f32" else 3000)
        c["batch"] = min(256, max(1, c["tokens"] // rng.choice([1, 7, 300])))
    return c


def _pairs(prefix: int, chunk: int) -> int:
    """Unmasked (query, key) pairs of a causal chunk on a prefix."""
    return chunk * prefix + chunk * (chunk + 1) // 2


def _ints(text: str) -> list:
    return [int(x) for x in text.split(",")]


def _lengths(case: dict) -> list:
    """The batch's context lengths: the case's own (its work does not depend on the seed)."""
    low, high, n = case["low"], case["high"], case["batch"]
    rng = random.Random(1000003 * n + 1009 * high + low)
    if case["lens"] == "fixed":
        return [high] * n
    if case["lens"] == "uniform":
        return [rng.randint(low, high) for _ in range(n)]
    mu = math.log(case.get("median") or math.sqrt(low * high))
    return [min(high, max(low, round(rng.lognormvariate(mu, 1.0)))) for _ in range(n)]


def _randn(shape, dtype, g) -> torch.Tensor:
    """N(0, 1) in `dtype`, made on the device (in pieces, so that no fp32 copy of a pool is kept)."""
    out = torch.empty(shape, dtype=dtype, device=DEVICE)
    flat, step = out.view(-1), 1 << 26
    for i in range(0, flat.numel(), step):
        part = flat[i:i + step]
        part.copy_(torch.randn(part.numel(), generator=g, device=DEVICE))
    return out


def _tables(lens: list, seed: int):
    """Block tables [B, max pages] (-1 padded, int32, on the device) and the pool's page count."""
    need = [(n + PAGE - 1) // PAGE for n in lens]
    total = sum(need)
    nb = total + total // 4 + 8
    perm = torch.randperm(nb, generator=torch.Generator().manual_seed(seed))[:total].to(torch.int32)
    table = torch.full((len(lens), max(need + [1])), -1, dtype=torch.int32)
    table[torch.arange(table.shape[1])[None, :] < torch.tensor(need)[:, None]] = perm
    return table.to(DEVICE), nb


def _int32(values) -> torch.Tensor:
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def _cumsum(values: list) -> list:
    out = [0]
    for v in values:
        out.append(out[-1] + v)
    return out


def _inputs(case: dict, seed: int) -> dict:
    """The case's inputs, by the seed alone (no code of the framework)."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dt, hq, hkv, d = DTYPES[case["dtype"]], case["hq"], case["hkv"], case["d"]
    s = {"case": case}
    if case["kind"] in ("decode", "decode_append", "gather"):
        lens = _lengths(case)
        random.Random(seed).shuffle(lens)
        s["lens"] = lens
        s["table"], nb = _tables(lens, seed)
        s["k_pool"] = _randn((nb, PAGE, hkv, d), dt, g)
        s["v_pool"] = _randn((nb, PAGE, hkv, d), dt, g)
        if case.get("outliers"):
            at = torch.rand(s["k_pool"].shape, generator=g, device=DEVICE) < case["outliers"]
            s["k_pool"] = torch.where(at, s["k_pool"] * 8, s["k_pool"])
        if case["kind"] == "gather":
            s["cu"], s["total"] = _int32(_cumsum(lens)), sum(lens)
        else:
            s["seq_lens"] = _int32(lens)
            s["max_len"] = max(lens)
            s["q"] = _randn((len(lens), hq, d), dt, g)
        if case["kind"] == "decode_append":
            s["k_new"] = _randn((len(lens), hkv, d), dt, g)
            s["v_new"] = _randn((len(lens), hkv, d), dt, g)
    elif case["kind"] == "prefill":
        chunks, prefixes = _ints(case["chunks"]), _ints(case["prefixes"])
        totals = [p + c for p, c in zip(prefixes, chunks)]
        s["table"], nb = _tables(totals, seed)
        # equal prefixes of whole pages are one cached prefix
        first = {}
        for i, p in enumerate(prefixes):
            if p and p % PAGE == 0:
                j = first.setdefault(p, i)
                s["table"][i, :p // PAGE] = s["table"][j, :p // PAGE]
        s["k_pool"] = _randn((nb, PAGE, hkv, d), dt, g)
        s["v_pool"] = _randn((nb, PAGE, hkv, d), dt, g)
        s["q"] = _randn((sum(chunks), hq, d), dt, g)
        s.update(chunks=chunks, totals=totals, cu=_int32(_cumsum(chunks)), seq_lens=_int32(totals),
                 max_q=max(chunks), max_len=max(totals))
    elif case["kind"] == "first_prefill":
        chunks = _ints(case["chunks"])
        cum = _cumsum(chunks)
        s["table"], s["pages"] = _tables(chunks, seed)
        s["q"] = _randn((cum[-1], hq, d), dt, g)
        s["k"] = _randn((cum[-1], hkv, d), dt, g)
        s["v"] = _randn((cum[-1], hkv, d), dt, g)
        s.update(chunks=chunks, max_q=max(chunks), cu=_int32(cum), num=_int32(chunks), start=_int32([0] * len(chunks)),
                 q_off=_int32([c * hq * d for c in cum[:-1]]), kv_off=_int32([c * hkv * d for c in cum[:-1]]))
    else:
        tokens, n = case["tokens"], case["batch"]
        rng = random.Random(1000003 * n + tokens)
        # one token for most sequences (decode), the rest of the tokens in a few chunks
        chunks = [1] * n
        for i in rng.sample(range(n), min(4, n)):
            chunks[i] += (tokens - n) // min(4, n)
        chunks[0] += tokens - sum(chunks)
        starts = [rng.randint(0, 1500) for _ in chunks]
        s["table"], nb = _tables([a + c for a, c in zip(starts, chunks)], seed)
        s["k_pool"] = torch.zeros((nb, PAGE, hkv, d), dtype=dt, device=DEVICE)
        s["v_pool"] = torch.zeros((nb, PAGE, hkv, d), dtype=dt, device=DEVICE)
        s["q"] = _randn((tokens, hq, d), dt, g)
        s["k"] = _randn((tokens, hkv, d), dt, g)
        s["v"] = _randn((tokens, hkv, d), dt, g)
        s.update(chunks=chunks, starts=starts, cu=_int32(_cumsum(chunks)), start=_int32(starts))
        pos = torch.cat([torch.arange(a, a + c) for a, c in zip(starts, chunks)]).double()
        angle = pos[:, None] * 10000.0 ** (-torch.arange(d // 2).double() * 2 / d)[None, :]
        s["cos"] = angle.cos().float().to(DEVICE)
        s["sin"] = angle.sin().float().to(DEVICE)
    return s


def prepare(case: dict, seed: int) -> dict:
    from lightllm_amd import kv_cache

    s = _inputs(case, seed)
    s["kc"] = kv_cache
    if case["kind"] == "first_prefill":
        s["pool"] = kv_cache.BlockAllocator(s["pages"], PAGE, case["hkv"], case["d"],
                                            kv_dtype=DTYPES[case["dtype"]], device=DEVICE)
    return s


def run(s: dict):
    kc, case = s["kc"], s["case"]
    kind = case["kind"]
    if kind == "decode":
        return kc.paged_decode(s["q"], s["k_pool"], s["v_pool"], s["table"], s["seq_lens"], s["max_len"],
                               num_splits=case["splits"])
    if kind == "decode_append":
        out = kc.paged_decode_append(s["q"], s["k_new"], s["v_new"], s["k_pool"], s["v_pool"], s["table"],
                                     s["seq_lens"], s["max_len"], num_splits=case["splits"])
        return out, s["k_pool"], s["v_pool"]
    if kind == "prefill":
        return kc.paged_prefill(s["q"], s["k_pool"], s["v_pool"], s["table"], s["cu"], s["seq_lens"],
                                s["max_q"], s["max_len"])
    if kind == "first_prefill":
        pool, n, total = s["pool"], len(s["chunks"]), s["q"].shape[0]
        kc.scatter_prefill_kv_batched(s["k"], s["v"], s["kv_off"], s["num"], s["start"], s["cu"], s["table"],
                                      s["table"].shape[1], n, total, pool)
        out = torch.empty_like(s["q"])
        kc.first_prefill_attn_batched(out, s["q"], s["k"], s["v"], case["hq"], case["hkv"], case["d"], s["q_off"],
                                      s["kv_off"], s["num"], s["cu"], s["start"], n, total,
                                      1.0 / math.sqrt(case["d"]), max_tokens=s["max_q"])
        return out, pool.k_storage, pool.v_storage
    if kind == "rope_append":
        slots = kc.build_slots(s["table"], s["cu"], s["start"], case["tokens"])
        kc.rope_append(s["q"], s["k"], s["v"], slots, s["cos"], s["sin"], s["k_pool"], s["v_pool"])
        return slots, s["q"], s["k"], s["k_pool"], s["v_pool"]
    return kc.gather_kv(s["k_pool"], s["v_pool"], s["table"], s["cu"], s["total"])


def work(case: dict) -> dict:
    es, hq, hkv, d = DTYPES[case["dtype"]].itemsize, case["hq"], case["hkv"], case["d"]
    row = hkv * d * es                      # one token's K (or V) row
    kind = case["kind"]
    if kind in ("decode", "decode_append"):
        toks, n = sum(_lengths(case)), case["batch"]
        extra = 4 * n * row if kind == "decode_append" else 0   # the new rows, in and out
        return {"bytes": 2 * toks * row + 2 * n * hq * d * es + toks // PAGE * 4 + 4 * n + extra,
                "flops": 4 * toks * hq * d}
    if kind == "gather":
        return {"bytes": 4 * sum(_lengths(case)) * row, "flops": 0}
    if kind == "rope_append":
        t = case["tokens"]
        return {"bytes": t * ((2 * hq + 5 * hkv) * d * es + 4 * d + 8), "flops": 3 * t * (hq + hkv) * d}
    chunks = _ints(case["chunks"])
    prefixes = _ints(case["prefixes"]) if kind == "prefill" else [0] * len(chunks)
    pairs = sum(_pairs(p, c) for p, c in zip(prefixes, chunks))
    shared = {p for p in prefixes if p % PAGE == 0}
    keys = sum(chunks) + sum(shared) + sum(p for p in prefixes if p % PAGE)
    nbytes = 2 * sum(chunks) * hq * d * es + 2 * keys * row
    if kind == "first_prefill":
        nbytes += 2 * keys * row            # the rows written to the pool
    return {"bytes": nbytes, "flops": 4 * pairs * hq * d}


def tolerance(case: dict):
    if case["kind"] == "gather":
        return "exact"
    if case["kind"] == "rope_append":
        # two products and one sum in 32 bits, rounded once to the rows' type
        return {"rel": {"f32": 1e-6, "f16": 1e-3, "bf16": 8e-3}[case["dtype"]]}
    # attention: 32-bit scores and sums; 16-bit types round the output, and prefill and
    # head_dim 256 the probabilities as well (four times the distance from exact() that was seen)
    return {"rel": {"f32": 1.6e-6, "f16": 1.2e-3, "bf16": 8.4e-3}[case["dtype"]]}


# ---------------------------------------------------------------------------------------------
# The same outputs in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------

def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, hist: int) -> torch.Tensor:
    """q [P, Hq, D], k and v [L, Hkv, D] -> [P, Hq, D]; query i sees keys up to hist + i."""
    p, hq, d = q.shape
    n, hkv = k.shape[0], k.shape[1]
    out = torch.empty((p, hq, d), dtype=torch.float64, device=q.device)
    hidden = torch.arange(n, device=q.device)[None, :] > hist + torch.arange(p, device=q.device)[:, None]
    for h in range(hkv):
        kt = k[:, h].double().t().contiguous()
        vh = v[:, h].double().contiguous()
        for j in range(h * (hq // hkv), (h + 1) * (hq // hkv)):
            s = torch.mm(q[:, j].double().contiguous(), kt) / math.sqrt(d)
            s.masked_fill_(hidden, -math.inf)
            out[:, j] = torch.mm(torch.softmax(s, dim=1), vh)
    return out


def _attend_one(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """One query token: q [Hq, D], k and v [L, Hkv, D] -> [Hq, D]."""
    hq, d = q.shape
    hkv = k.shape[1]
    kk = k.double().permute(1, 0, 2).contiguous()              # [Hkv, L, D]
    vv = v.double().permute(1, 0, 2).contiguous()
    qq = q.double().view(hkv, hq // hkv, d)
    out = torch.empty((hkv, hq // hkv, d), dtype=torch.float64, device=q.device)
    for j in range(hq // hkv):
        p = torch.softmax((kk * qq[:, j, None, :]).sum(-1) / math.sqrt(d), dim=1)
        out[:, j] = (p[:, :, None] * vv).sum(1)
    return out.view(hq, d)


def _rows(pool: torch.Tensor, table: torch.Tensor, n: int) -> torch.Tensor:
    pages = table[:(n + PAGE - 1) // PAGE].long()
    return pool[pages].reshape(-1, pool.shape[2], pool.shape[3])[:n]


def _slots(table: torch.Tensor, seqs: list, positions: list) -> torch.Tensor:
    table = table.cpu().long()
    pos = torch.tensor(positions)
    return (table[torch.tensor(seqs), pos // PAGE] * PAGE + pos % PAGE).to(DEVICE)


def _put(pool: torch.Tensor, slots: torch.Tensor, rows: torch.Tensor) -> None:
    pool.view(-1, pool.shape[2], pool.shape[3])[slots] = rows


def exact(case: dict, seed: int):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "gather":
        return tuple(torch.cat([_rows(s[p], s["table"][i], n) for i, n in enumerate(s["lens"])])
                     for p in ("k_pool", "v_pool"))
    if kind in ("decode", "decode_append"):
        lens = s["lens"]
        if kind == "decode_append":
            slots = _slots(s["table"], list(range(len(lens))), [n - 1 for n in lens])
            _put(s["k_pool"], slots, s["k_new"])
            _put(s["v_pool"], slots, s["v_new"])
        out = torch.stack([_attend_one(s["q"][i], _rows(s["k_pool"], s["table"][i], n),
                                       _rows(s["v_pool"], s["table"][i], n)) for i, n in enumerate(lens)])
        return out if kind == "decode" else (out, s["k_pool"], s["v_pool"])
    if kind == "rope_append":
        seqs = [i for i, c in enumerate(s["chunks"]) for _ in range(c)]
        positions = [a + t for a, c in zip(s["starts"], s["chunks"]) for t in range(c)]
        slots = _slots(s["table"], seqs, positions)
        half = case["d"] // 2
        cos, sin = s["cos"].double()[:, None, :], s["sin"].double()[:, None, :]
        turned = []
        for x in (s["q"].double(), s["k"].double()):
            a, b = x[..., :half], x[..., half:]
            turned.append(torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1))
        k_pool = s["k_pool"].double()
        _put(k_pool, slots, turned[1])
        _put(s["v_pool"], slots, s["v"])
        return slots, turned[0], turned[1], k_pool, s["v_pool"]
    cum = _cumsum(s["chunks"])
    if kind == "first_prefill":
        out = torch.cat([_attend(s["q"][a:b], s["k"][a:b], s["v"][a:b], 0) for a, b in zip(cum, cum[1:])])
        shape = (s["pages"], PAGE, case["hkv"], case["d"])
        pools = [torch.zeros(shape, dtype=s["k"].dtype, device=DEVICE) for _ in range(2)]
        seqs = [i for i, c in enumerate(s["chunks"]) for _ in range(c)]
        slots = _slots(s["table"], seqs, [t for c in s["chunks"] for t in range(c)])
        for pool, rows in zip(pools, (s["k"], s["v"])):
            _put(pool, slots, rows)
        return out, pools[0], pools[1]
    out = []
    for i, (a, b) in enumerate(zip(cum, cum[1:])):
        n = s["totals"][i]
        out.append(_attend(s["q"][a:b], _rows(s["k_pool"], s["table"][i], n),
                           _rows(s["v_pool"], s["table"][i], n), n - (b - a)))
    return torch.cat(out)
