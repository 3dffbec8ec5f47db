"""Attention backward with few workgroups: query streams and key ranges dealt out to up to 16 workgroups, some of them with one tile or
none, or to a workgroup's wavefronts (fp32).  Gradients against float64 autograd over the plain chain."""
import math

import pytest
import torch

import tinytorch_amd as tt

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# relative error (2-norm) of a gradient: P, dS, the saved output and the result are rounded to the type once each
# (4 roundings of 2^-24, 2^-11, 2^-8), dP - delta cancels up to some ten times that; fp32: hardware exp2 besides
REL = {"f32": 1e-5, "f16": 5e-3, "bf16": 3e-2}


def grads(go, q, k, v, hidden, bias):
    q, k, v = (t.double().requires_grad_() for t in (q, k, v))
    G, D = q.shape[1] // k.shape[1], q.shape[3]
    s = torch.matmul(q, k.repeat_interleave(G, 1).transpose(-1, -2).contiguous()) / math.sqrt(D)
    s = (s if bias is None else s + bias.double()).masked_fill(hidden, -math.inf)
    out = torch.matmul(torch.softmax(s, -1), v.repeat_interleave(G, 1))
    out.backward(go.double())
    return out.detach(), q.grad, k.grad, v.grad


def run(B, Hq, Hkv, L, S, D, dtype, mode):
    g = torch.Generator(device="cuda").manual_seed(L * 7 + S + D)
    q, go = (torch.randn(B, Hq, L, D, generator=g, device="cuda").to(DT[dtype]) for _ in "qg")
    k, v = (torch.randn(B, Hkv, S, D, generator=g, device="cuda").to(DT[dtype]) for _ in "kv")
    keys, rows = torch.arange(S, device="cuda"), torch.arange(L, device="cuda")
    hidden, bias, kw = torch.zeros(L, S, dtype=torch.bool, device="cuda"), None, {}
    if mode == "top-left" or mode == "bottom-right":
        hidden = keys[None] > rows[:, None] + (S - L if mode == "bottom-right" else 0)
        kw = dict(isCausal=True, causalAlign=mode)
    elif mode == "bool":
        seen = torch.rand(Hq, L, S, generator=g, device="cuda") < 0.4
        seen[..., S // 2] = True
        hidden, kw = ~seen, dict(attnMask=seen)
    elif mode == "add":
        bias = torch.randn(L, S, generator=g, device="cuda").to(DT[dtype])
        kw = dict(attnMask=bias)
    elif mode == "lens":
        lens = torch.tensor([max(1, S // 3)] * (B - 1) + [S], device="cuda", dtype=torch.int32)
        hidden, kw = (keys[None] >= lens[:, None]).view(B, 1, 1, S), dict(kvLens=lens)
    ref = grads(go, q, k, v, hidden, bias)
    out = tt.sdpAttention(q, k, v, **kw)
    got = (out,) + tuple(tt.sdpAttentionBackward(go, q, k, v, out, **kw))
    for name, x, y in zip(("out", "dq", "dk", "dv"), got, ref):
        rel = ((x.double() - y).norm() / y.norm()).item()
        assert rel <= REL[dtype], (name, rel)


# one tile and less, tiles around 32 and 128, grouped heads (one stream of many short ones), long streams of one head
SIZES = [(1, 1, 1, 3, 5), (1, 4, 4, 128, 128), (2, 4, 1, 33, 31), (1, 2, 2, 129, 200), (2, 8, 2, 97, 65), (1, 1, 1, 700, 900), (1, 7, 1, 260, 257)]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("mode", ["full", "top-left", "bottom-right", "bool", "add", "lens"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "B%dH%dk%dL%dS%d" % s)
def test_gradients(size, mode, D, dtype):
    B, Hq, Hkv, L, S = size
    if mode == "bottom-right" and S < L:
        pytest.skip("rows without keys")
    run(B, Hq, Hkv, L, S, D, dtype, mode)


@pytest.mark.parametrize("dtype,D", [("f32", 4), ("f32", 40), ("f32", 96), ("f32", 124), ("f16", 8), ("f16", 48), ("bf16", 80), ("f16", 120)])
@pytest.mark.parametrize("mode", ["full", "top-left", "bool", "lens"])
def test_between_the_kernels_sizes(dtype, D, mode):
    run(2, 4, 2, 150, 190, D, dtype, mode)
    run(1, 2, 1, 600, 800, D, dtype, mode)
