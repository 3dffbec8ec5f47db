"""Rows that no key gives any weight, one rule for every kernel: a batch entry without keys gives zeros (the reference's empty
contraction), a row whose scores are all -inf gives NaN (its softmax's 0 / 0), whole or with the keys divided, whatever the route."""
import math

import pytest
import torch

import tinytorch_amd as tt

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def operands(seed, B, Hq, Hkv, L, S, D, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(B, h, n, D, generator=g, device="cuda").to(DT[dtype]) for h, n in ((Hq, L), (Hkv, S), (Hkv, S))]


# decode whole and split, few rows per KV head, short rows (128-row tiles whole and split), 256-row tiles whole and split
SHAPES = [(2, 8, 2, 1, 40), (2, 8, 2, 1, 1500), (1, 4, 4, 3, 700), (1, 2, 1, 12, 333), (2, 4, 4, 100, 200), (1, 2, 2, 100, 2000),
          (2, 4, 2, 300, 300), (1, 2, 1, 300, 4096), (8, 32, 32, 100, 1100)]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("D", [64, 72, 128, 90])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_scores_of_minus_infinity(shape, D, dtype):
    B, Hq, Hkv, L, S = shape
    print("weightless", shape, D, dtype, flush=True)
    q, k, v = operands(1, B, Hq, Hkv, L, S, D, dtype)
    q[..., 0] = 1.0
    k[B - 1, Hkv - 1, :, 0] = -math.inf  # every score of these rows
    lens = torch.full((B,), S, dtype=torch.int32, device="cuda")
    for kw in ({}, {"kvLens": lens}, {"kvLens": lens, "isCausal": True, "causalAlign": "bottom-right"}):
        out = tt.sdpAttention(q, k, v, **kw)
        nan = torch.zeros(B, Hq, dtype=torch.bool, device="cuda")
        nan[B - 1, Hq - Hq // Hkv:] = True
        assert torch.equal(out.isnan().all(-1).all(-1), nan) and torch.equal(out.isnan().any(-1).any(-1), nan), kw


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("D", [64, 72, 128, 90])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_no_keys(shape, D, dtype):
    B, Hq, Hkv, L, S = shape
    q, k, v = operands(2, B, Hq, Hkv, L, S, D, dtype)
    lens = torch.full((B,), S, dtype=torch.int32, device="cuda")
    lens[0] = 0
    for causal in (False, True):
        out = tt.sdpAttention(q, k, v, kvLens=lens, isCausal=causal, causalAlign="bottom-right")
        assert torch.count_nonzero(out[0]).item() == 0 and not out.isnan().any()


@pytest.mark.parametrize("D", [64, 128])
def test_fewer_keys_than_rows(D):
    """Bottom-right alignment with fewer keys than rows starts at the first key: every row sees one (a call of 300 (batch, head)
    pairs, whose split depends on its size)."""
    B, H, L, S = 15, 20, 128, 1024
    q, k, v = operands(3, B, H, H, L, S, D, "bf16")
    lens = torch.full((B,), S, dtype=torch.int32, device="cuda")
    lens[3], lens[7] = 100, 1
    out = tt.sdpAttention(q, k, v, kvLens=lens, isCausal=True, causalAlign="bottom-right")
    for b, n in ((3, 100), (7, 1)):
        s = torch.matmul(q[b].double(), k[b, :, :n].double().transpose(-1, -2).contiguous()) / math.sqrt(D)
        s = s.masked_fill(torch.arange(n, device="cuda")[None] > torch.arange(L, device="cuda")[:, None], -math.inf)
        ref = torch.matmul(torch.softmax(s, -1), v[b, :, :n].double())
        assert ((out[b].double() - ref).norm() / ref.norm()).item() <= 8e-3
