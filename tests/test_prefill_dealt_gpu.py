"""Attention on workgroups of 128 rows whose keys are dealt out to two groups of wavefronts (sdpa_prefill_dealt.hip): row tiles and
halves of 32 keys that end anywhere, a group without keys, both alignments of the diagonal, more rows than keys, pages, key counts,
divided keys, and maxima that rise.  The whole output against float64."""
import numpy as np
import pytest
import torch

from gpu_util import call, make_inputs
from tinytorch_amd import _capi
from tinytorch_amd.function import build_params

pytestmark = pytest.mark.gpu

# Relative error (2-norm) of correct results: probabilities and results rounded to the type once, about 0.4 of its epsilon each.
REL = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def reference(q, k, v, causal, align, lens):
    B, Hq, L, D = q.shape
    S, G = k.shape[2], Hq // k.shape[1]
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    for b in range(B):
        n = S if lens is None else int(lens[b])
        if n == 0:
            continue
        kk, vv = k[b, :, :n].double().repeat_interleave(G, 0), v[b, :, :n].double().repeat_interleave(G, 0)
        s = q[b].double() @ kk.transpose(-1, -2).contiguous() / D ** 0.5
        if causal:
            off = max(0, n - L) if align == "bottom-right" else 0
            s = s.masked_fill(torch.arange(n, device="cuda")[None] > torch.arange(L, device="cuda")[:, None] + off, float("-inf"))
        out[b] = torch.softmax(s, -1) @ vv
    return out


def check(case, dtype, D, mul=1.0, page=0, lens=None, entries=("forward", "prefill")):
    B, Hq, Hkv, L, S, causal, align = case
    _, (q, k, v) = make_inputs(311 + L + S + D, B, Hq, Hkv, L, S, D, dtype, mul)
    kw = dict(causal=causal, align=align, kv_lens=None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda"))
    ref = reference(q, k, v, causal, align, lens)
    kp, vp = k, v
    if page:
        per = -(-S // page)
        table = torch.from_numpy(np.random.default_rng(L).permutation(B * per).astype(np.int32)).cuda().view(B, per)
        kp, vp = (torch.zeros(B * per, Hkv, page, D, dtype=q.dtype, device="cuda") for _ in "kv")
        for b in range(B):
            for e in range(per):
                for pool, rows in ((kp, k), (vp, v)):
                    part = rows[b, :, e * page:(e + 1) * page]
                    pool[int(table[b, e]), :, :part.shape[1]] = part
        kw["block_table"] = table
        kw["kv_lens"] = torch.tensor([S] * B if lens is None else lens, dtype=torch.int32, device="cuda")
    p = build_params(q, kp, vp, torch.empty_like(q), causal, None, None, kw["kv_lens"], align, kw.get("block_table"))
    assert _capi.kernel(p) == "dealt", _capi.kernel(p)
    for entry in entries:
        out = torch.full_like(q, 7.0)
        rc, out = call(entry, q, kp, vp, out=out, **kw)
        assert rc == 0
        err = ((out.double() - ref).norm() / ref.norm()).item()
        assert err <= REL[dtype], (entry, err)


TL, BR = "top-left", "bottom-right"
CASES = [
    # B, Hq, Hkv, L, S, causal, align
    (8, 16, 8, 129, 129, True, TL),      # a second row tile of one row; a group without a key on the diagonal's first rows
    (8, 16, 8, 160, 160, True, TL),
    (8, 16, 16, 150, 161, True, BR),     # the diagonal inside a half
    (2, 8, 2, 513, 513, False, TL),      # 17 halves: the second group one fewer, its last one whole
    (4, 8, 8, 514, 545, False, TL),      # a last half of one key
    (8, 16, 16, 256, 290, False, TL),
    (1, 16, 4, 700, 650, True, TL),      # rows beyond the last key
    (1, 16, 4, 650, 700, True, TL),
    (1, 16, 4, 650, 700, True, BR),
    (1, 32, 4, 1001, 1001, True, TL),
    (1, 4, 2, 700, 5000, True, BR),      # divided keys
    (1, 4, 2, 1100, 3000, True, BR),
]


@pytest.mark.parametrize("D,dtype", [(128, "bf16"), (128, "f16"), (64, "f16"), (64, "bf16")])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%dH%dk%dL%dS%d-c%d-%s" % c)
def test_against_float64(case, D, dtype):
    check(case, dtype, D)


@pytest.mark.parametrize("page,case,lens", [
    (64, (3, 8, 2, 600, 1500, True, BR), None),
    (64, (3, 8, 2, 600, 1500, True, BR), [1500, 0, 601]),
    (128, (3, 4, 2, 700, 3000, True, BR), [3000, 1999, 705]),   # divided
    (64, (1, 4, 2, 1100, 9000, True, BR), None),                # three windows of the block table
])
def test_pages_and_key_counts(page, case, lens):
    check(case, "bf16", 128, page=page, lens=lens)


@pytest.mark.parametrize("D", [128, 64])
def test_key_counts_without_pages(D):
    check((4, 8, 8, 514, 545, True, BR), "f16", D, lens=[545, 1, 0, 33])
    check((4, 8, 8, 514, 545, False, TL), "f16", D, lens=[545, 1, 0, 64])


@pytest.mark.parametrize("D", [128, 64])
def test_maxima_that_rise(D):
    """Scores with a standard deviation of 5 to 9: the exponentials' maximum is raised on the way, differently in the two groups, and a
    row's weights lie on a few keys."""
    check((1, 16, 4, 650, 700, True, BR), "f16", D, mul=0.8 * (1024 / D) ** 0.25)


def test_weightless_rows_and_no_finite_neighbours():
    """Keys that hold infinities beyond a row's diagonal do not reach it; rows before them stay finite."""
    _, (q, k, v) = make_inputs(5, 1, 16, 4, 650, 650, 128, "bf16")
    rc, clean = call("forward", q, k, v, causal=True)
    assert rc == 0
    k2, v2 = k.clone(), v.clone()
    k2[:, :, 600:] = float("inf")
    v2[:, :, 600:] = float("nan")
    rc, out = call("forward", q, k2, v2, causal=True)
    assert rc == 0
    assert torch.equal(out[:, :, :512], clean[:, :, :512])
    assert torch.isfinite(out[:, :, :576]).all()
