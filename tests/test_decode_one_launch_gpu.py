"""Decode calls whose sequences' keys are one workgroup's, four or eight wavefronts of it (plan_decode): key counts around a wavefront's 32
keys and the workgroup's turns, every number of query rows and width of a value row (the sums over a chunk's lanes differ with it),
pages and key counts.  Against float64."""
import ctypes

import pytest
import torch

from gpu_util import call, make_inputs
from tinytorch_amd import _capi
from tinytorch_amd.function import build_params

pytestmark = pytest.mark.gpu

REL = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 2e-6}  # one rounding of the result; fp32: sums of up to 1000 products


def check(B, Hq, Hkv, S, D, dtype, lens=None, page=0, one_launch=False):
    _, (q, k, v) = make_inputs(31 * S + D + Hq, B, Hq, Hkv, 1, S, D, dtype)
    kv = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda")
    table, kp, vp = None, k, v
    if page:
        per = -(-S // page)
        table = torch.randperm(B * per, generator=torch.Generator().manual_seed(S)).to(torch.int32).cuda().view(B, per)
        kp, vp = (torch.zeros(B * per, Hkv, page, D, dtype=q.dtype, device="cuda") for _ in "kv")
        for b in range(B):
            for e in range(per):
                n = min(page, S - e * page)
                kp[int(table[b, e]), :, :n], vp[int(table[b, e]), :, :n] = k[b, :, e * page:e * page + n], v[b, :, e * page:e * page + n]
        kv = torch.tensor([S] * B if lens is None else lens, dtype=torch.int32, device="cuda")
    p = build_params(q, kp, vp, torch.empty_like(q), False, None, None, kv, "top-left", table)
    if one_launch:
        assert _capi.lib().ttsdpa_workspace_bytes(ctypes.byref(p)) == 0
    rc, out = call("decode", q, kp, vp, kv_lens=kv, block_table=table) if dtype != "f32" else call("forward", q, kp, vp, kv_lens=kv, block_table=table)
    assert rc == 0
    ref = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    for b in range(B):
        n = S if lens is None else lens[b]
        for h in range(Hq):
            if n:
                g = h * Hkv // Hq
                ref[b, h] = torch.softmax(q[b, h].double() @ k[b, g, :n].double().t().contiguous() / D ** 0.5, -1) @ v[b, g, :n].double()
    err = ((out.double() - ref).norm() / ref.norm()).item()
    assert err <= REL[dtype], err


@pytest.mark.parametrize("D,dtype", [(128, "bf16"), (64, "f16"), (80, "bf16"), (128, "f32"), (64, "f32")])
@pytest.mark.parametrize("G", [1, 3, 5, 8])
@pytest.mark.parametrize("S", [256, 257, 289])
def test_rows_and_widths(S, G, D, dtype):
    check(2, 2 * G, 2, S, D, dtype, one_launch=S == 256)


@pytest.mark.parametrize("S", [1, 31, 33, 130, 255])
def test_few_keys(S):
    check(3, 4, 2, 256, 128, "f16", lens=[S, 0, 256])


@pytest.mark.parametrize("page", [0, 32, 64])
@pytest.mark.parametrize("D,dtype", [(128, "bf16"), (64, "f16"), (64, "f32")])
def test_many_pairs(page, D, dtype):
    """More (sequence, KV head) pairs than half of the CUs: 1000 keys in one launch too."""
    lens = [1000 - 37 * b for b in range(24)]
    lens[5], lens[7] = 0, 1
    check(24, 16, 8, 1000, D, dtype, lens=lens, page=page, one_launch=True)
