"""Edges of single kernel variants and of the rules that choose them (remainders, smallest
sizes, special values), against plain torch or the CPU oracle."""
import numpy as np
import pytest
import torch

from lightllm_amd import kv_cache as kc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rot", [64, 36], ids=["vector", "scalar"])
def test_bf16_rounding_of_every_kind_of_value(rot):
    """fp32 -> bf16 in the kernels: nearest even, ties, overflow to infinity, denormals, signed
    zeros, infinities and NaN as torch rounds them on the CPU.  With q = (1, 0) pairs a rotation's
    first output is exactly its cosine, so the cosine table carries the values."""
    g = torch.Generator().manual_seed(7)
    half, T = rot // 2, 64
    bits = torch.randint(0, 2**32, (T, half), generator=g, dtype=torch.int64).to(torch.uint32).view(torch.float32)
    cos = bits.clone()
    edge = torch.tensor([0.0, -0.0, 1.0, 1.00390625, 1.01171875, -1.00390625, 3.4028235e38, -3.4028235e38,
                         3.3895e38, 1e-40, -1e-40, 9.2e-41, 1.1754944e-38, float("inf"), float("-inf"),
                         float("nan")])
    cos[0, :16] = edge
    sin = torch.zeros(T, half)
    q = torch.zeros(T, 1, 64, dtype=torch.bfloat16)
    q[:, :, :half] = 1.0
    k, v = torch.zeros(T, 1, 64, dtype=torch.bfloat16), torch.zeros(T, 1, 64, dtype=torch.bfloat16)
    pool = torch.zeros(8, 16, 1, 64, dtype=torch.bfloat16, device=DEV)
    qd = q.to(DEV)
    kc.rope_append(qd, k.to(DEV), v.to(DEV), torch.full((T,), -1, device=DEV), cos.to(DEV), sin.to(DEV),
                   pool, pool.clone())
    got = qd.cpu()[:, 0, :half]
    want = cos.to(torch.bfloat16)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert np.array_equal(got[~nan].view(torch.int16).numpy(), want[~nan].view(torch.int16).numpy())


def _attend64(q, k, v, hist):
    """Causal attention in float64 on the CPU: q [P, Hq, D], k, v [L, Hkv, D]."""
    q, k, v = q.double(), k.double(), v.double()
    g = q.shape[1] // k.shape[1]
    kk, vv = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    s = torch.einsum("phd,lhd->hpl", q, kk) / q.shape[2] ** 0.5
    s.masked_fill_(torch.arange(k.shape[0])[None, None, :] > hist + torch.arange(q.shape[0])[None, :, None],
                   float("-inf"))
    return torch.einsum("hpl,lhd->phd", torch.softmax(s, -1), vv)


# fp32 prefill by terms (head_dim 64, 96, 128): tile remainders, large and small values and
# infinities, mostly in launches that cut nothing (test_prefill_f32_terms_cut has the cuts).
SPLIT = ["plain", "k_one_large", "k_minus_inf", "v_one_inf", "v_tiny", "k_tiny_q_large", "k_large_window",
         "v_zero"]


@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("case", SPLIT)
def test_prefill_f32_split_terms(case, d):
    g = torch.Generator().manual_seed(len(case) + d)
    hq, hkv, P, L = 4, 2, 133, 4300 if case == "k_large_window" else 333
    hist = L - P
    q = torch.randn(P, hq, d, generator=g)
    k = torch.randn(L, hkv, d, generator=g)
    v = torch.randn(L, hkv, d, generator=g)
    unit = 1.0
    if case == "k_one_large":       # tile 1: |k| beyond the fp16 terms, the scores moderate
        q[..., 3] *= 1e-4
        k[70, :, 3] = 3.0e4
    elif case == "k_minus_inf":     # the key drops out of the softmax
        q[..., 5] = q[..., 5].abs() + 0.1
        k[100, 0, 5] = float("-inf")
    elif case == "v_one_inf":       # a key that every row sees
        v[40, 1, 7] = float("inf")
    elif case == "v_tiny":
        unit = 1e-6
        v *= unit
    elif case == "k_tiny_q_large":
        k *= 1e-4
        q *= 1e4
    elif case == "k_large_window":  # past one window of staged page ids, in K and in V
        q[..., 3] *= 1e-4
        k[4200, :, 3] = -3.0e4
        v[4160:4170] *= 1e3
        unit = 1e3
    elif case == "v_zero":
        v.zero_()
        k[:64] = 0
    nb = (L + 15) // 16
    perm = torch.randperm(nb, generator=g)
    kp, vp = torch.zeros(nb, 16, hkv, d), torch.zeros(nb, 16, hkv, d)
    pos = torch.arange(L)
    kp[perm[pos // 16], pos % 16], vp[perm[pos // 16], pos % 16] = k, v
    ref = _attend64(q, k, v, hist)
    cu, lens = torch.tensor([0, P], dtype=torch.int32, device=DEV), torch.tensor([L], dtype=torch.int32, device=DEV)
    dev = [t.to(DEV) for t in (q, kp, vp)]
    table = perm.to(torch.int32).reshape(1, -1).to(DEV)
    outs = {"split": kc.paged_prefill(*dev, table, cu, lens, P, L).cpu().double(),
            "unsplit": kc.paged_prefill(*dev, table, cu, lens, P, L,
                                        workspace=torch.empty(0, dtype=torch.uint8, device=DEV)).cpu().double()}
    if hist < L and case in ("plain", "k_one_large", "v_tiny", "v_zero"):   # the contiguous form: rows 0 .. P - 1
        off = torch.zeros(1, dtype=torch.int32, device=DEV)
        out = torch.empty_like(dev[0])
        kc.first_prefill_attn_batched(out, dev[0], k[:P].contiguous().to(DEV), v[:P].contiguous().to(DEV), hq, hkv, d,
                                      off, off, torch.tensor([P], dtype=torch.int32, device=DEV), cu, off, 1, P,
                                      d ** -0.5, max_tokens=P)
        first = _attend64(q, k[:P], v[:P], 0)
        assert torch.all((out.cpu().double() - first).abs() <= 1e-6 * unit + 1e-5 * first.abs())
    fine = torch.isfinite(ref)
    for name, out in outs.items():
        assert torch.equal(torch.isfinite(out), fine), (case, name)
        assert torch.equal(out[~fine], ref[~fine]), (case, name)
        err = (out - ref)[fine].abs()
        assert torch.all(err <= 1e-6 * unit + 1e-5 * ref[fine].abs()), (case, name, float(err.max()))


# The same with cut key ranges (35 tiles in chunks of 7), with values on both sides of what the
# terms hold (2^-60 .. 2^60; other tiles run on the fp32 matrix instructions) in the first tile of
# a later chunk (keys 448 ..) and inside one (keys 576 ..), and finite values of any size and of
# mixed sizes, whose dims are each as exact as dims of one.
TERMS = ["plain", "k_beyond", "k_minus_inf", "k_tiny_q_large", "v_beyond", "v_edge", "v_1e35", "v_one_inf",
         "v_tiny", "v_mixed_dims", "v_zero"]


@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("case", TERMS)
def test_prefill_f32_terms_cut(case, d):
    g = torch.Generator().manual_seed(len(case) + d)
    hq, hkv, P, L = 4, 2, 133, 2200
    q = torch.randn(P, hq, d, generator=g)
    k = torch.randn(L, hkv, d, generator=g)
    v = torch.randn(L, hkv, d, generator=g)
    unit = torch.ones(d, dtype=torch.float64)
    if case == "k_beyond":
        q[..., 3] *= 1e-20
        k[450, :, 3] = 3e20
        k[600, :, 3] = -2e20
    elif case == "k_minus_inf":     # the keys drop out of the softmax
        q[..., 5] = q[..., 5].abs() + 0.1
        k[450, 0, 5] = k[600, 1, 5] = float("-inf")
    elif case == "k_tiny_q_large":
        k *= 1e-20
        q *= 1e20
    elif case == "v_beyond":
        v[450:460] *= 1e30
        v[600] *= 1e30
        unit *= 1e30
    elif case == "v_edge":
        v[450], v[600] = 2.0 ** 60, 2.0 ** 60 * (1 + 2.0 ** -23)
        unit *= 2.0 ** 60
    elif case == "v_1e35":
        v *= 1e35
        unit *= 1e35
    elif case == "v_one_inf":       # keys that every row sees
        v[450, 1, 7] = float("inf")
        v[600, 0, 9] = float("-inf")
    elif case == "v_tiny":
        v *= 1e-25
        unit *= 1e-25
    elif case == "v_mixed_dims":
        unit = 10.0 ** -(torch.arange(d) % 12).double()
        v *= unit.float()
    elif case == "v_zero":
        v.zero_()
        k[448:512] = 0
    nb = (L + 15) // 16
    perm = torch.randperm(nb, generator=g)
    kp, vp = torch.zeros(nb, 16, hkv, d), torch.zeros(nb, 16, hkv, d)
    pos = torch.arange(L)
    kp[perm[pos // 16], pos % 16], vp[perm[pos // 16], pos % 16] = k, v
    assert kc.lib().llkv_paged_prefill_workspace_size(1, P, P, L, hq, d, 16, kc.dtype_code(q.dtype)) > 0
    cu, lens = torch.tensor([0, P], dtype=torch.int32, device=DEV), torch.tensor([L], dtype=torch.int32, device=DEV)
    out = kc.paged_prefill(q.to(DEV), kp.to(DEV), vp.to(DEV), perm.to(torch.int32).reshape(1, -1).to(DEV), cu, lens,
                           P, L).cpu().double()
    ref = _attend64(q, k, v, L - P)
    fine = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(out), fine)
    assert torch.equal(out[~fine], ref[~fine])
    bar = 1e-6 * unit + 1e-5 * ref.abs()
    assert torch.all(((out - ref).abs() <= bar)[fine]), float(((out - ref).abs() / bar)[fine].max())


# 2-norm errors against 64 bits: 1e-6 is 17 roundings of 2^-24; the row sum and the output take one
# per 64-key tile (24 tiles), at random sizes and signs, and the fp32 matrix instructions' own
# summation is 5e-7 off.  Dims of 1e-4 .. 1e-10 beside dims of one, K with a constant large dim (scores
# of 112, of which 2^-24 is 7e-6), a few rows.
@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (4, 4, 96), (8, 2, 128)])
def test_prefill_f32_holds_32_bits(hq, hkv, d):
    def run(P, L, change, dims=slice(None)):
        g = torch.Generator().manual_seed(P + L)
        q, k, v = (torch.randn(n, h, d, generator=g) for n, h in ((P, hq), (L, hkv), (L, hkv)))
        change(q, k, v)
        nb = (L + 15) // 16
        kp, vp = torch.zeros(nb * 16, hkv, d), torch.zeros(nb * 16, hkv, d)
        kp[:L], vp[:L] = k, v
        ids = torch.arange(nb, dtype=torch.int32).reshape(1, -1)
        out = kc.paged_prefill(q.to(DEV), kp.view(nb, 16, hkv, d).to(DEV), vp.view(nb, 16, hkv, d).to(DEV), ids.to(DEV),
                               torch.tensor([0, P], dtype=torch.int32, device=DEV),
                               torch.tensor([L], dtype=torch.int32, device=DEV), P, L).cpu().double()[..., dims]
        ref = _attend64(q, k, v, L - P)[..., dims]
        return float(torch.linalg.vector_norm(out - ref) / torch.linalg.vector_norm(ref))

    def dim7(scale):
        def change(q, k, v):
            v[..., 7] *= scale
        return change

    def biased(q, k, v):
        k[..., 3] += 300 * d ** 0.5 / 8
        q[..., 3] = 3

    for scale in (1.0, 1e-4, 1e-6, 1e-10):
        assert run(150, 1500, dim7(scale), dims=7) <= 1e-6, scale
    # five rows on nothing: at most five keys, so the roundings are those of a score (D / 16 at its
    # full size, 2^-24 each at random) and of single products: the fp32 instructions give 7.1e-8 .. 8.1e-8
    assert run(5, 5, dim7(1.0)) <= 8.1e-8
    assert run(150, 1500, biased) <= 3e-5


# Work items of a prefill launch: (prefixes, chunks) with cut key ranges (one long sequence: many
# chunks; several of uneven length; the merge's rows past a chunk's query rows), more units than
# the ranking's 32 per pass, more than it ranks at all, and sequences without rows or keys.
def _items(name):
    g = torch.Generator().manual_seed(11)
    if name == "one_long":
        return 4, 2, [40000], [5]
    if name == "uneven":
        return 4, 2, [6000, 0, 1500, 16], [3, 140, 129, 1]
    if name == "units_300":
        return 2, 1, torch.randint(0, 900, (300,), generator=g).tolist(), torch.randint(0, 3, (300,), generator=g).tolist()
    if name == "units_1100":
        return 2, 1, torch.randint(0, 90, (1100,), generator=g).tolist(), torch.randint(0, 3, (1100,), generator=g).tolist()
    return 4, 2, [0, -7, 2000, 0, -64], [0, 7, 130, 40, 64]   # "no_keys": keys = prefix + chunk = 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("name", ["one_long", "uneven", "units_300", "units_1100", "no_keys"])
def test_prefill_work_items(name, dtype):
    g = torch.Generator().manual_seed(12)
    d = 64
    hq, hkv, prefixes, chunks = _items(name)
    totals = [p + c for p, c in zip(prefixes, chunks)]
    need = [(n + 15) // 16 for n in totals]
    nb = sum(need) + 1
    kp = torch.randn(nb, 16, hkv, d, generator=g).to(dtype)
    vp = torch.randn(nb, 16, hkv, d, generator=g).to(dtype)
    q = torch.randn(sum(chunks), hq, d, generator=g).to(dtype)
    perm = torch.randperm(nb, generator=g).to(torch.int32)
    table = torch.full((len(chunks), max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    cu = torch.tensor([0] + torch.tensor(chunks).cumsum(0).tolist(), dtype=torch.int32)
    out = kc.paged_prefill(q.to(DEV), kp.to(DEV), vp.to(DEV), table.to(DEV), cu.to(DEV),
                           torch.tensor(totals, dtype=torch.int32, device=DEV), max(chunks), max(totals)).cpu().double()
    for i, (n, c) in enumerate(zip(totals, chunks)):
        if c == 0:
            continue
        got = out[cu[i]:cu[i + 1]]
        if n == 0:
            assert torch.all(got == 0), i
            continue
        rows = table[i, :need[i]].long()
        k, v = (p[rows].reshape(-1, hkv, d)[:n] for p in (kp, vp))
        ref = _attend64(q[cu[i]:cu[i + 1]], k, v, n - c)
        bar = 2e-3 * (ref.abs() + ref.square().mean(-1, keepdim=True).sqrt()) if dtype == torch.float16 else \
            1e-6 + 1e-5 * ref.abs()
        assert torch.all((got - ref).abs() <= bar), (i, float(((got - ref).abs() / bar).max()))


# How a launch cuts key ranges, from the chunk counts that it leaves for the merge kernel in the
# workspace's last slot (one query block per chunk here, so unit n is sequence n): one long unit fills
# the GPU in chunks of at least 8 tiles; batches whose longest unit is near a compute unit's share are
# not cut; kernels of one work-group per CU take as many chunks as run at once.
CUTS = [
    ("one_unit", torch.float16, 32, 32, 96, [66], [3381], [7]),              # 54 tiles: seven of eight
    ("one_unit_d256", torch.float16, 16, 8, 256, [63], [4125], [9]),         # 66 tiles: nine
    ("near_share", torch.float16, 32, 8, 128, [128] * 7, [1100] * 6 + [1500], None),
    ("long_beside_short", torch.float16, 32, 8, 128, [3, 40], [200, 2000], [1, 4]),   # 32 tiles
    ("one_round", torch.float32, 16, 8, 256, [128] * 6, [1031, 1159, 1287, 1415, 1543, 1671], [2, 2, 3, 3, 3, 3]),
]


@pytest.mark.parametrize("name,dtype,hq,hkv,d,chunks,prefixes,want", CUTS, ids=[c[0] for c in CUTS])
def test_prefill_cut_counts(name, dtype, hq, hkv, d, chunks, prefixes, want):
    totals = [p + c for p, c in zip(prefixes, chunks)]
    n, width = len(chunks), (max(totals) + 15) // 16
    pool = torch.zeros(width, 16, hkv, d, dtype=dtype, device=DEV)
    table = torch.arange(width, dtype=torch.int32, device=DEV).repeat(n, 1)
    q = torch.zeros(sum(chunks), hq, d, dtype=dtype, device=DEV)
    cu = torch.tensor([0] + torch.tensor(chunks).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    size = kc.lib().llkv_paged_prefill_workspace_size(n, sum(chunks), max(chunks), max(totals), hq, d, 16,
                                                      kc.dtype_code(dtype))
    ws = torch.full((size,), 255, dtype=torch.uint8, device=DEV)
    out = kc.paged_prefill(q, pool, pool, table, cu, torch.tensor(totals, dtype=torch.int32, device=DEV),
                           max(chunks), max(totals), workspace=ws)
    assert torch.all(out == 0)
    slot = hq * 128 * (1 + d) * 4
    counts = ws[size - slot:size - slot + 8 * n].view(torch.int32)[1::2].tolist()
    if want is None:
        assert all(c in (-1, 1) for c in counts), counts   # -1: the host did not let it cut
    else:
        assert counts == want


# Balanced decode: a unit cut into exactly the merge's four entries per trip, fewer, more, and many
# (one sequence of nearly all pages), beside short sequences inside one share.
@pytest.mark.parametrize("d,hq,hkv", [(64, 14, 2), (128, 32, 8), (256, 16, 8)])
@pytest.mark.parametrize("long", [2000, 9000, 30000])
def test_balanced_merge_entries(long, d, hq, hkv):
    g = torch.Generator().manual_seed(long + d)
    B = 520 // hkv
    lens = torch.randint(1, 200, (B,), generator=g).tolist()
    lens[B // 2] = long
    assert kc.decode_schedule(B, hq, hkv, d, long, torch.float16)[0] == "balanced"
    need = [(n + 15) // 16 for n in lens]
    nb = sum(need)
    kp = torch.randn(nb, 16, hkv, d, generator=g).half()
    vp = torch.randn(nb, 16, hkv, d, generator=g).half()
    q = torch.randn(B, hq, d, generator=g).half()
    perm = torch.randperm(nb, generator=g).to(torch.int32)
    table = torch.full((B, max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    out = kc.paged_decode(q.to(DEV), kp.to(DEV), vp.to(DEV), table.to(DEV),
                          torch.tensor(lens, dtype=torch.int32, device=DEV), long).cpu().double()
    for i in (0, 1, B // 2 - 1, B // 2, B // 2 + 1, B - 1):
        rows = table[i, :need[i]].long()
        k, v = (p[rows].reshape(-1, hkv, d)[:lens[i]] for p in (kp, vp))
        ref = _attend64(q[i:i + 1], k, v, lens[i] - 1)[0]
        bar = 2e-3 * (ref.abs() + ref.square().mean(-1, keepdim=True).sqrt())
        assert torch.all((out[i] - ref).abs() <= bar), (i, float(((out[i] - ref).abs() / bar).max()))


# Streaming loads: batches of more than 192 MB by their lengths, every instantiation that has them.
# The host takes the kernels that may stream by the bound; a bound below 192 MB (the lengths may be
# beyond it) gives the plain ones, with the same schedule and work-groups, and the same bits.  In
# "half_shared" the sequences of one half read the other's pages, which are not streamed.
STREAM = [
    ("f16_d128", 40, 32, 8, 128, torch.float16, "balanced", False),
    ("bf16_d128_half_shared", 70, 28, 4, 128, torch.bfloat16, "balanced", True),
    ("f16_d64", 160, 14, 2, 64, torch.float16, "balanced", False),
    ("bf16_d64", 60, 8, 8, 64, torch.bfloat16, "balanced", False),
    ("f32_d64", 170, 14, 2, 64, torch.float32, "balanced", False),
    ("f32_d96", 34, 8, 8, 96, torch.float32, "balanced", False),
    ("f32_d256", 34, 16, 8, 256, torch.float32, "balanced", False),
    ("f16_d256", 34, 8, 8, 256, torch.float16, "balanced", False),
    ("bf16_d256_half_shared", 36, 16, 8, 256, torch.bfloat16, "balanced", True),
    ("f16_d64_wide", 16, 14, 2, 64, torch.float16, "unit", False),
    ("bf16_d64_wide_half_shared", 18, 14, 2, 64, torch.bfloat16, "unit", True),
]


@pytest.mark.parametrize("name,B,hq,hkv,d,dtype,sched,shared", STREAM, ids=[s[0] for s in STREAM])
def test_decode_streaming_loads(name, B, hq, hkv, d, dtype, sched, shared):
    g = torch.Generator().manual_seed(len(name))
    row = hkv * d * 2 * dtype.itemsize
    limit = (192 << 20) // (B * row)   # tokens per sequence at the rule
    long = int(1.35 * limit * B / (B - 5))
    lens = torch.randint(long - long // 10, long, (B,), generator=g).tolist()
    lens[:5] = [1, 16, 17, 0, 33]
    low, high = limit - 16, long       # the bounds on both sides of the rule
    assert sum(lens) * row > 200 << 20 and B * low * row < 192 << 20
    assert kc.decode_schedule(B, hq, hkv, d, low, dtype) == kc.decode_schedule(B, hq, hkv, d, high, dtype)
    assert kc.decode_schedule(B, hq, hkv, d, high, dtype)[0] == sched
    need = [(n + 15) // 16 for n in lens]
    nb = sum(need) + 1
    gd = torch.Generator(device=DEV).manual_seed(len(name))
    kp, vp = (torch.randn(nb, 16, hkv, d, generator=gd, device=DEV).to(dtype) for _ in range(2))
    q, kn, vn = (torch.randn(B, h, d, generator=gd, device=DEV).to(dtype) for h in (hq, hkv, hkv))
    perm = torch.randperm(nb, generator=g).to(torch.int32)
    table = torch.full((B, max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    if shared:   # every page but the last two
        for i in range(B // 2, B - 1, 2):
            n = min(need[i], need[i + 1]) - 2
            table[i + 1, :n] = table[i, :n]
    td, ld = table.to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV)
    slots = torch.tensor([int(table[i, (n - 1) // 16]) * 16 + (n - 1) % 16 if n else -1 for i, n in enumerate(lens)],
                         device=DEV)
    pools = [(kp.clone(), vp.clone()) for _ in range(2)]
    # append, then decode; the fused call gives the same bits, and so do the plain kernels
    kc.append_kv(kn, vn, slots, *pools[0])
    out = kc.paged_decode(q, *pools[0], td, ld, high)
    fused = kc.paged_decode_append(q, kn, vn, *pools[1], td, ld, high)
    assert torch.equal(out, fused) and all(torch.equal(a, b) for a, b in zip(*pools))
    assert torch.equal(out, kc.paged_decode(q, *pools[0], td, ld, low))
    assert torch.equal(out, kc.paged_decode_append(q, kn, vn, *pools[1], td, ld, low))
    for i in list(range(6)) + [B // 2, B - 2, B - 1]:
        if lens[i] == 0:
            assert torch.all(out[i] == 0)
            continue
        rows = table[i, :need[i]].long().to(DEV)
        k, v = (p[rows].reshape(-1, hkv, d)[:lens[i]].cpu() for p in pools[0])
        ref = _attend64(q[i:i + 1].cpu(), k, v, lens[i] - 1)[0]
        rms = ref.square().mean(-1, keepdim=True).sqrt()
        bar = {torch.float32: 1e-6 + 1e-5 * ref.abs(), torch.float16: 2e-3 * (ref.abs() + rms),
               torch.bfloat16: 1.6e-2 * (ref.abs() + rms)}[dtype]
        err = (out[i].cpu().double() - ref).abs()
        assert torch.all(err <= bar), (i, float((err / bar).max()))


def test_decode_shared_prefix_stays_cached():
    """Pages that several sequences read are not streamed past the caches: a batch on one prefix
    takes at most 1.12 times the plain kernels' time (streamed, 1.3 times).  Both in turn, the
    fastest of each; the bound chooses the kernels as in test_decode_streaming_loads."""
    B, hq, hkv, d, prefix = 40, 32, 8, 128, 4096
    lens = [prefix + 17 + 3 * i for i in range(B)]
    need = [(n + 15) // 16 for n in lens]
    table = torch.full((B, max(need)), -1, dtype=torch.int32)
    at = prefix // 16
    for i, n in enumerate(need):
        table[i, :prefix // 16] = torch.arange(prefix // 16)
        table[i, prefix // 16:n] = torch.arange(at, at + n - prefix // 16)
        at += n - prefix // 16
    pools = [torch.randn(at, 16, hkv, d, device=DEV).half() for _ in range(2)]
    q = torch.randn(B, hq, d, device=DEV).half()
    td, ld = table.to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV)
    bounds = [(192 << 20) // (B * hkv * d * 4) - 16, max(lens)]
    assert all(kc.decode_schedule(B, hq, hkv, d, b, q.dtype)[0] == "balanced" for b in bounds)
    best, outs = [float("inf")] * 2, [None] * 2
    for _ in range(8):
        for i, bound in enumerate(bounds):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            outs[i] = kc.paged_decode(q, *pools, td, ld, bound)
            a.record()
            for _ in range(20):
                kc.paged_decode(q, *pools, td, ld, bound)
            b.record()
            b.synchronize()
            best[i] = min(best[i], a.elapsed_time(b))
    assert torch.equal(*outs)
    assert best[1] <= 1.12 * best[0], best


def test_decode_streaming_choice_under_capture():
    """A captured fused append + decode under a bound beyond the streaming rule follows the lengths of
    each replay: beyond 192 MB, far below, and beyond again, with eager work between."""
    B, hq, hkv, d, long = 40, 32, 8, 128, 1700
    nb = B * ((long + 15) // 16)
    pools = [torch.randn(nb, 16, hkv, d, device=DEV).half() for _ in range(2)]
    q, kn, vn = (torch.randn(B, h, d, device=DEV).half() for h in (hq, hkv, hkv))
    table = torch.randperm(nb, device=DEV).to(torch.int32).reshape(B, -1)
    lens = torch.full((B,), long, dtype=torch.int32, device=DEV)
    assert B * long * hkv * d * 4 > 192 << 20 and kc.decode_schedule(B, hq, hkv, d, long, q.dtype)[0] == "balanced"
    ws = torch.empty(kc.decode_workspace_bytes(B, hq, hkv, d, 16, long), dtype=torch.uint8, device=DEV)
    out = torch.empty_like(q)
    step = lambda o, p: kc.paged_decode_append(q, kn, vn, *p, table, lens, long, out=o, workspace=ws)
    step(out, pools)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(out, pools)
    for n in (long, 33, long - 5):
        lens.fill_(n)
        eager = [p.clone() for p in pools]
        want = step(torch.empty_like(q), eager)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and all(torch.equal(a, b) for a, b in zip(pools, eager)), n


@pytest.mark.parametrize("extra", [0, 5])
def test_gather_streaming_edge(extra):
    """Gathers on both sides of the streaming rule (4 x rows x row bytes at 288 MB), bit for bit."""
    hkv, d = 8, 128
    n = (288 << 20) // (4 * hkv * d * 2) + extra
    g = torch.Generator(device=DEV).manual_seed(5)
    lens = [n // 3, n - n // 3 - 1, 1]
    need = [(x + 15) // 16 for x in lens]
    nb = sum(need) + 2
    kp = torch.randint(0, 1 << 15, (nb, 16, hkv, d), generator=g, device=DEV, dtype=torch.int16).view(torch.float16)
    vp = torch.randint(0, 1 << 15, (nb, 16, hkv, d), generator=g, device=DEV, dtype=torch.int16).view(torch.float16)
    perm = torch.randperm(nb, generator=torch.Generator().manual_seed(6)).to(torch.int32).to(DEV)
    table = torch.full((3, max(need)), -1, dtype=torch.int32, device=DEV)
    at, rows = 0, []
    for i, m in enumerate(need):
        table[i, :m] = perm[at:at + m]
        rows.append((perm[at:at + m].long()[:, None] * 16 + torch.arange(16, device=DEV)).reshape(-1)[:lens[i]])
        at += m
    cu = torch.tensor([0, lens[0], lens[0] + lens[1], n], dtype=torch.int32, device=DEV)
    k, v = kc.gather_kv(kp, vp, table, cu, n)
    rows = torch.cat(rows)
    for got, pool in ((k, kp), (v, vp)):
        assert torch.equal(got.view(torch.int16), pool.view(torch.int16).view(-1, hkv, d)[rows])
