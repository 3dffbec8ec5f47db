"""Key splits of the 4-wavefront prefill kernels (16-bit and fp32): calls with few row tiles divide their keys among workgroups.  The
call with its workspace against float64 and, where the unsplit kernel can be asked for the same call, against that: every
kernel size and the head sizes between them, masks (rows that see nothing, the type's lowest value), causal alignments,
per-batch key counts, grouped heads, strided queries."""
import ctypes
import math

import pytest
import torch

import tinytorch_amd as tt
from tinytorch_amd import _capi
from tinytorch_amd.function import build_params

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# relative error of the whole output (2-norm): the probabilities' and the result's rounding to the type (2^-11, 2^-8), of random sign,
# at most once each; fp32: sums of up to 1500 products and the hardware's exp2 (some 2^-22)
REL = {"f32": 5e-6, "f16": 1e-3, "bf16": 8e-3}


def reference(q, k, v, causal=None, mask=None, lens=None):
    B, H, L, D = q.shape
    S, G = k.shape[2], H // k.shape[1]
    k, v = (t.double().repeat_interleave(G, 1) for t in (k, v))
    s = torch.matmul(q.double(), k.transpose(-1, -2).contiguous()) / math.sqrt(D)
    if mask is not None:
        s = s.masked_fill(~mask, -math.inf) if mask.dtype == torch.bool else s + mask.double()
    keys, rows = torch.arange(S, device="cuda"), torch.arange(L, device="cuda")
    n = torch.full((B,), S, device="cuda") if lens is None else lens.long()
    hidden = keys[None, None, :] >= n[:, None, None]
    if causal:
        off = (n - L) if causal == "bottom-right" else torch.zeros_like(n)
        hidden = hidden | (keys[None, None, :] > rows[None, :, None] + off[:, None, None])
    s = s.masked_fill(hidden[:, None].expand(B, H, L, S) if hidden.shape[1] == L else hidden[:, None], -math.inf)
    return torch.matmul(torch.softmax(s, -1), v)


def check(got, ref, dtype):
    assert torch.equal(got.isnan(), ref.isnan())
    rel = ((got.double() - ref).nan_to_num().norm() / ref.nan_to_num().norm()).item()
    assert rel <= REL[dtype], rel


def operands(seed, B, Hq, Hkv, L, S, D, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(B, h, n, D, generator=g, device="cuda").to(DT[dtype]) for h, n in ((Hq, L), (Hkv, S), (Hkv, S))]


def splits(q, k, v, **kw):
    p = build_params(q, k, v, torch.empty_like(q), kw.get("causal", False), kw.get("mask"), None, kw.get("lens"), kw.get("align", "top-left"), None)
    return _capi.lib().ttsdpa_workspace_bytes(ctypes.byref(p)) > 0


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("D", [8, 32, 64, 80, 96, 120, 128, 160, 192, 256])
@pytest.mark.parametrize("causal", [False, True])
def test_head_sizes(D, causal, dtype):
    if dtype == "f32" and D > 128:
        pytest.skip("fp32 of more than 128 columns: the general kernel")
    for B, Hq, Hkv, L, S in ((1, 2, 1, 127, 777), (1, 3, 3, 129, 640), (2, 4, 1, 65, 1000)):
        q, k, v = operands(D + L, B, Hq, Hkv, L, S, D, dtype)
        align = "bottom-right" if causal else "top-left"
        check(tt.sdpAttention(q, k, v, isCausal=causal, causalAlign=align), reference(q, k, v, causal and align), dtype)
        if not causal and L == 127 and D <= 128 and dtype != "f32":
            assert splits(q, k, v)


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("kind", ["keys", "rows", "add", "lowest"])
@pytest.mark.parametrize("S", [449, 900])
def test_masks(S, kind, dtype):
    B, H, L, D = 2, 3, 449, 64
    q, k, v = operands(S, B, H, H, L, S, D, dtype)
    g = torch.Generator(device="cuda").manual_seed(3)
    if kind == "keys":
        mask = (torch.arange(S, device="cuda")[None] < torch.tensor([[S], [70]], device="cuda")).view(B, 1, 1, S)
    elif kind == "rows":  # rows that see nothing, one key in the last split, everything
        mask = torch.rand(L, S, generator=g, device="cuda") < 0.5
        mask[5], mask[7], mask[8] = False, False, True
        mask[7, S - 1] = True
    elif kind == "add":
        mask = torch.randn(H, L, S, generator=g, device="cuda").to(DT[dtype])
    else:  # whole splits at the type's lowest value
        mask = torch.zeros(L, S, device="cuda", dtype=DT[dtype])
        mask[:, :S - 10] = torch.finfo(DT[dtype]).min
    assert splits(q, k, v, mask=mask) or dtype == "f32"  # (fp32: dealt out to the wavefronts)
    check(tt.sdpAttention(q, k, v, attnMask=mask), reference(q, k, v, mask=mask), dtype)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("D", [64, 72])
def test_key_counts_and_strides(D, dtype):
    B, Hq, Hkv, L, S = 3, 4, 2, 100, 900
    g = torch.Generator(device="cuda").manual_seed(1)
    qkv = torch.randn(B, L, Hq, D, generator=g, device="cuda").to(DT[dtype])
    q = qkv.transpose(1, 2)
    k, v = operands(2, B, Hq, Hkv, L, S, D, dtype)[1:]
    lens = torch.tensor([900, 0, 130], device="cuda", dtype=torch.int32)
    for causal in (False, True):
        got = tt.sdpAttention(q, k, v, isCausal=causal, kvLens=lens, causalAlign="bottom-right")
        assert torch.count_nonzero(got[1]).item() == 0
        ref = reference(q, k, v, causal and "bottom-right", None, lens)
        check(got[::2], ref[::2], dtype)
