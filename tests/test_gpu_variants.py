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
