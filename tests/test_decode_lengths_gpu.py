"""Decode over sequences of different lengths: each sequence's keys are divided over all of its splits, in units of 128 keys, and the
splits of neighbouring sequences begin at different XCDs; lengths around those units, empty sequences, pages."""
import math

import pytest
import torch

import tinytorch_amd as tt

pytestmark = pytest.mark.gpu

# relative error (2-norm): the result's rounding, and probabilities in fp32
REL = {torch.float32: 5e-6, torch.float16: 1e-3, torch.bfloat16: 8e-3}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("page", [0, 64])
@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(9, 4, 1, 1500, 128), (40, 8, 4, 2100, 64), (3, 8, 8, 300, 128), (130, 2, 2, 520, 64)])
def test_lengths(B, Hq, Hkv, S, D, page, dtype):
    g = torch.Generator(device="cuda").manual_seed(B)
    q = torch.randn(B, Hq, 1, D, generator=g, device="cuda").to(dtype)
    k, v = (torch.randn(B, Hkv, S, D, generator=g, device="cuda").to(dtype) for _ in "kv")
    edges = [S, 0, 1, 127, 128, 129, 255, 256, 257]
    lens = [edges[i] if i < len(edges) and edges[i] <= S else 1 + (i * 977) % S for i in range(B)]
    n = torch.tensor(lens, dtype=torch.int32, device="cuda")
    if page:
        per = -(-S // page)
        table = torch.randperm(B * per, generator=g, device="cuda").to(torch.int32).view(B, per)
        pools = []
        for t in (k, v):
            pool = torch.full((B * per, Hkv, page, D), float("nan"), dtype=dtype, device="cuda")
            whole = torch.full((B, Hkv, per * page, D), float("nan"), dtype=dtype, device="cuda")
            whole[:, :, :S] = t
            pool[table.long().view(-1)] = whole.view(B, Hkv, per, page, D).transpose(1, 2).reshape(B * per, Hkv, page, D)
            pools.append(pool)
        got = tt.sdpAttention(q, *pools, kvLens=n, blockTable=table)
    else:
        got = tt.sdpAttention(q, k, v, kvLens=n)
    kd, vd = (t.double().repeat_interleave(Hq // Hkv, 1) for t in (k, v))
    s = (q.double() * kd).sum(-1) / math.sqrt(D)
    s = s.masked_fill(torch.arange(S, device="cuda")[None, None] >= n[:, None, None], -math.inf)
    ref = (torch.softmax(s, -1).nan_to_num()[..., None] * vd).sum(-2, keepdim=True)
    assert torch.count_nonzero(got[n == 0]) == 0
    assert ((got.double() - ref).norm() / ref.norm()).item() <= REL[dtype]
