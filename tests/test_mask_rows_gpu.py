"""Query rows at the ends of what an attnMask can say: every key at the type's lowest value or at another value far beyond the
scores, where the biased scores of a row round to one number and the reference's chain is a plain softmax of equal scores;
values that differ out there; and, in the backward, rows whose keys are all hidden.  At key counts of both parities, the kernels' sizes and the sizes
between them, whole and with the keys or rows divided among workgroups or wavefronts."""
import math

import pytest
import torch

import tinytorch_amd as tt

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# relative error of a whole result (2-norm): what the probabilities' and the result's rounding to the type leave (2^-11, 2^-8, at most once
# each and once more in a gradient); fp32: sums of up to 1000 products and the hardware's exp2 (some 2^-22).  A biased score is an fp32
# number in every kernel: near fp16's lowest value, -65504, its steps are 2^-8, so that such a row's weights are off by up to
# 2^-9 each, of random sign.
REL = {"f32": 5e-6, "f16": 1e-3 + 2 ** -9, "bf16": 8e-3}


def operands(seed, B, Hq, Hkv, L, S, D, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(B, h, n, D, generator=g, device="cuda").to(DT[dtype]) for h, n in ((Hq, L), (Hkv, S), (Hkv, S), (Hq, L))]


def additive(L, S, dtype, seed=1):
    """Rows in turn: all keys at the lowest value; all at one far value; the lowest but for one key; ordinary values; the lowest and a
    far value in turn (only the latter count); ordinary ones again with one key far above the others."""
    low = torch.finfo(DT[dtype]).min
    far = -6e4 if dtype == "f16" else -1e9
    g = torch.Generator(device="cuda").manual_seed(seed)
    m = torch.randn(L, S, generator=g, device="cuda")
    m[0::6] = low
    m[1::6] = far
    m[2::6] = low
    m[2::6, S - 1] = 0.0
    m[4::6] = low
    m[4::6, 0::3] = -4e4 if dtype == "f16" else -1e37
    m[5::6, S // 2] = 3e4 if dtype == "f16" else 2e38
    return m.to(DT[dtype])


def probabilities(q, k, mask, lens=None):
    """softmax of the biased scores, which are fp32 numbers as in the reference's chain; the sums in 64 bits."""
    B, H, L, D = q.shape
    S = k.shape[2]
    k = k.double().repeat_interleave(H // k.shape[1], 1)
    s = torch.matmul(q.double(), k.transpose(-1, -2).contiguous()) / math.sqrt(D)
    if mask.dtype == torch.bool:
        s = s.masked_fill(~mask, -math.inf)
    else:
        s = (s.float() + mask.float()).double()
    if lens is not None:
        s = s.masked_fill((torch.arange(S, device="cuda")[None] >= lens[:, None])[:, None, None], -math.inf)
    return torch.softmax(s, -1)


def rel_err(got, ref):
    return ((got.double() - ref).nan_to_num().norm() / ref.nan_to_num().norm()).item()


def forward_reference(q, k, v, p):
    return torch.matmul(p, v.double().repeat_interleave(q.shape[1] // v.shape[1], 1))


def backward_reference(q, k, v, g, p):
    """dq, dk, dv; rows whose keys are all hidden (probabilities NaN) weigh nothing."""
    G = q.shape[1] // k.shape[1]
    p = p.nan_to_num(0.0)
    kk, vv, qd, gd = k.double().repeat_interleave(G, 1), v.double().repeat_interleave(G, 1), q.double(), g.double()
    out = torch.matmul(p, vv)
    dp = torch.matmul(gd, vv.transpose(-1, -2).contiguous())
    ds = p * (dp - (gd * out).sum(-1, keepdim=True)) / math.sqrt(q.shape[-1])
    group = lambda t: t.view(t.shape[0], k.shape[1], G, *t.shape[2:]).sum(2)
    return torch.matmul(ds, kk), group(torch.matmul(ds.transpose(-1, -2).contiguous(), qd)), group(torch.matmul(p.transpose(-1, -2).contiguous(), gd))


# (B, Hq, Hkv, L, S): one short row tile; more than 128 rows (the pipelined kernel at head_dim 128); keys divided among workgroups
SHAPES = [(2, 4, 2, 37, 197), (2, 4, 2, 37, 200), (1, 4, 2, 150, 333), (1, 4, 2, 150, 332), (1, 2, 1, 100, 901)]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("D", [32, 64, 80, 128, 90, 160])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward_far_values(shape, D, dtype):
    print("far values", shape, D, dtype, flush=True)
    B, Hq, Hkv, L, S = shape
    q, k, v, _ = operands(sum(shape) + D, B, Hq, Hkv, L, S, D, dtype)
    mask = additive(L, S, dtype)
    got = tt.sdpAttention(q, k, v, attnMask=mask)
    assert not got.isnan().any()
    assert rel_err(got, forward_reference(q, k, v, probabilities(q, k, mask))) <= REL[dtype]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_forward_far_values_beside_key_counts(dtype):
    B, H, L, S, D = 3, 4, 70, 203, 64
    q, k, v, _ = operands(5, B, H, H, L, S, D, dtype)
    lens = torch.tensor([203, 66, 1], device="cuda", dtype=torch.int32)
    mask = additive(L, S, dtype)
    got = tt.sdpAttention(q, k, v, attnMask=mask, kvLens=lens)
    ref = forward_reference(q, k, v, probabilities(q, k, mask, lens))
    assert not got.isnan().any()
    assert rel_err(got, ref) <= REL[dtype]


def check_backward(q, k, v, g, mask, dtype, lens=None):
    out = tt.sdpAttention(q, k, v, attnMask=mask, kvLens=lens)
    grads = tt.sdpAttentionBackward(g, q, k, v, out, attnMask=mask, kvLens=lens)
    refs = backward_reference(q, k, v, g, probabilities(q, k, mask, lens))
    for name, got, ref in zip(("dq", "dk", "dv"), grads, refs):
        assert not got.isnan().any(), name
        assert rel_err(got, ref) <= REL[dtype], (name, rel_err(got, ref))
    return grads


# as above; few rows or keys for the wavefronts to share; enough of both that nothing is divided
BACKWARD_SHAPES = SHAPES + [(1, 1, 1, 20, 33), (4, 16, 16, 260, 333)]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("D", [64, 80, 128, 90, 160])
@pytest.mark.parametrize("shape", BACKWARD_SHAPES, ids=str)
def test_backward_far_values(shape, D, dtype):
    print("backward, far values", shape, D, dtype, flush=True)
    B, Hq, Hkv, L, S = shape
    q, k, v, g = operands(sum(shape) + D, B, Hq, Hkv, L, S, D, dtype)
    check_backward(q, k, v, g, additive(L, S, dtype), dtype)


@pytest.mark.parametrize("kind", ["bool", "add"])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("D", [64, 80, 128, 90])
@pytest.mark.parametrize("shape", BACKWARD_SHAPES, ids=str)
def test_backward_hidden_rows(shape, D, dtype, kind):
    """The forward's own output (NaN in such rows) goes back in: dq is 0 there, dk and dv hold the other rows' sums."""
    print("backward, hidden rows", shape, D, dtype, kind, flush=True)
    B, Hq, Hkv, L, S = shape
    q, k, v, g = operands(sum(shape) + D, B, Hq, Hkv, L, S, D, dtype)
    seen = torch.rand(L, S, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda") < 0.6
    seen[:, S // 2] = True
    seen[3::7] = False
    seen[L - 1] = False
    mask = seen if kind == "bool" else torch.zeros(L, S, device="cuda", dtype=DT[dtype]).masked_fill(~seen, -math.inf)
    assert tt.sdpAttention(q, k, v, attnMask=mask)[:, :, 3::7].isnan().all()
    dq = check_backward(q, k, v, g, mask, dtype)[0]
    assert torch.count_nonzero(dq[:, :, 3::7]).item() == 0


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("S", [203, 204])
def test_backward_hidden_rows_beside_key_counts(S, dtype):
    B, H, L, D = 3, 4, 70, 64
    q, k, v, g = operands(6, B, H, H, L, S, D, dtype)
    lens = torch.tensor([S, 66, 1], device="cuda", dtype=torch.int32)
    seen = torch.rand(L, S, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda") < 0.6
    seen[5], seen[6, :66] = False, False
    _, dk, dv = check_backward(q, k, v, g, seen, dtype, lens)
    assert torch.count_nonzero(dk[1, :, 66:]).item() == 0 and torch.count_nonzero(dv[2, :, 1:]).item() == 0
