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


# fp32 prefill by two fp16 terms (head_dim 64, 96, 128): tile remainders, and tiles that do not fit
# the two terms (they run on the fp32 matrix instructions), at the edges of the rule: one value
# beyond 2^9, infinities, whole tensors too small, q too large.
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
