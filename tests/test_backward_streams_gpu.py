"""The 16-bit backward pair's streams and splits (sdpa_backward_d128.hip, backward_splits_16bit): key counts around its tiles of 32 and
its two steps at a time, query streams of few tiles, row tiles whose wavefronts end at different tiles, maxima that rise on the way, and numbers of splits
that are no power of two over more workgroups than run side by side.  All three gradients against float64."""
import ctypes

import pytest
import torch

from gpu_util import backward_call, call, make_inputs
from tinytorch_amd import _capi
from tinytorch_amd.function import build_backward_params

pytestmark = pytest.mark.gpu

# Relative error (2-norm) of correct results: P and dS rounded to the type for their products and the gradients once more, each about
# 0.3 of its epsilon; the forward's rounded output enters delta.
REL = {"f16": 2.0 ** -10, "bf16": 2.0 ** -7}


def reference(q, k, v, go, causal, off):
    G = q.shape[1] // k.shape[1]
    grads = [torch.zeros_like(t, dtype=torch.float64) for t in (q, k, v)]
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            qd, kd, vd, gd = q[b, h].double(), k[b, h // G].double(), v[b, h // G].double(), go[b, h].double()
            s = qd @ kd.t().contiguous() / q.shape[3] ** 0.5
            if causal:
                s = s.masked_fill(torch.arange(k.shape[2], device="cuda")[None] > torch.arange(q.shape[2], device="cuda")[:, None] + off, float("-inf"))
            p = torch.softmax(s, -1)
            dp = gd @ vd.t().contiguous()
            ds = p * (dp - (p * dp).sum(-1, keepdim=True)) / q.shape[3] ** 0.5
            grads[0][b, h] += ds @ kd
            grads[1][b, h // G] += ds.t().contiguous() @ qd
            grads[2][b, h // G] += p.t().contiguous() @ gd
    return grads


def check(case, dtype, D, mul=1.0, rel=1.0):
    B, Hq, Hkv, L, S, causal, align = case
    _, (q, k, v) = make_inputs(17 + L + S, B, Hq, Hkv, L, S, D, dtype, mul)
    _, (go, _, _) = make_inputs(18 + L + S, B, Hq, Hkv, L, S, D, dtype)
    rc, out = call("forward", q, k, v, causal=causal, align=align)
    assert rc == 0
    grads = [torch.empty_like(t) for t in (q, k, v)]
    p = build_backward_params(q, k, v, out, go, *grads, causal, None, None, None, align)
    assert _capi.backward_kernel(p) == "other"
    rc, got = backward_call(q, k, v, out, go, causal, None, None, None, align, grads)
    assert rc == 0
    for name, x, ref in zip(("dq", "dk", "dv"), got, reference(q, k, v, go, causal, max(0, S - L) if align == "bottom-right" else 0)):
        err = ((x.double() - ref).norm() / ref.norm()).item()
        assert err <= rel * REL[dtype], (name, err)


TL, BR = "top-left", "bottom-right"


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("case", [
    (1, 16, 4, 1100, 1100, True, TL),
    (2, 4, 4, 1056, 1056, True, TL),      # whole tiles
    (1, 8, 2, 1025, 1057, True, BR),      # one row, one key beyond whole tiles
    (1, 8, 8, 1060, 95, False, TL),       # three tiles, the last one ragged
    (1, 8, 8, 1060, 160, False, TL),      # five whole ones
    (1, 8, 8, 1060, 33, False, TL),
    (1, 8, 8, 1100, 200, True, TL),       # rows beyond the last key
    (1, 8, 4, 200, 1500, True, BR),
    (2, 2, 1, 129, 2111, False, TL),      # divided key ranges
], ids=lambda c: "B%dH%dk%dL%dS%d-c%d-%s" % c)
def test_dq_stream(case, dtype):
    check(case, dtype, 128)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("Hq,Hkv", [(6, 2), (5, 5), (7, 1)])
@pytest.mark.parametrize("L", [33, 64, 96, 160, 193])
def test_dkv_stream_of_few_tiles(L, Hq, Hkv, dtype):
    """Fewer tiles than the ring's stages, none for the second group of wavefronts, one left over, a ragged one at either end; key
    blocks that do not end with the keys."""
    check((1, Hq, Hkv, L, 1230, False, TL), dtype, 128)
    check((1, Hq, Hkv, L, 1230, True, BR), dtype, 128)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_maxima_that_rise(dtype):
    """Scores with a standard deviation of 7: the running maximum is raised within the streams."""
    check((1, 8, 4, 1100, 1100, True, TL), dtype, 128, mul=0.8 * (1024 / 128) ** 0.25, rel=2.0)  # (dS differs from its sum's terms by more)


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("case", [(4, 56, 8, 383, 383, True, TL), (4, 32, 4, 909, 909, True, TL), (2, 32, 8, 700, 700, True, TL)],
                         ids=lambda c: "B%dH%dk%dL%dS%d-c%d-%s" % c)
def test_splits_of_a_key_block_walk_alike(case, D):
    """Causal calls of a multiple of eight (batch, KV head) pairs, whose workgroups walk their tiles in alternating directions."""
    check(case, "bf16", D)
