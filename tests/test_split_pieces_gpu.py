"""Split prefill calls over caches whose sequences have lengths of their own, contiguous and paged: every piece of every row tile is
taken once, whatever the lengths, and tables longer than what a wavefront holds of them (64 entries) are walked through.
Launches of the 4-wavefront kernels number up to 256 pieces (1024 with one row tile a head) by division; the cases that name a
number of pieces have more than that and search the sequences' lengths, as the pipelined kernel always does.
Against float64."""
import ctypes

import pytest
import torch

import tinytorch_amd as tt
from test_paged_cache_gpu import scatter_to_pages
from test_tile_splits_gpu import check, operands, reference
from tinytorch_amd import _capi
from tinytorch_amd.function import build_params

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, L, S, D, dtype, page, lengths (None: S)
    (1, 2, 1, 300, 13000, 128, "bf16", 64, None),        # 204 entries of the table; the pipelined kernel
    (2, 2, 1, 257, 9000, 128, "f16", 128, [9000, 4097]),
    (3, 4, 2, 260, 4500, 128, "bf16", 64, [4500, 0, 1]),
    (70, 1, 1, 130, 2200, 128, "f16", 256, "spread"),     # more sequences than lanes
    (20, 7, 7, 20, 700, 64, "f16", 64, "spread"),         # the 4-wavefront kernel
    (3, 8, 2, 9, 3000, 64, "bf16", 64, [3000, 64, 1500]),  # grouped heads share row tiles
    (5, 4, 1, 140, 1500, 64, "f32", 64, "spread"),
    (30, 4, 4, 200, 3000, 64, "bf16", 256, "spread", 256),
    (12, 7, 7, 129, 2500, 80, "f16", 64, "spread", 256),
    (342, 1, 1, 20, 30000, 32, "bf16", 4096, "spread", 1024),
]


def pieces(q, k, v, causal, align, lens, table=None):
    """Pieces of the call's launch, from its records: 32 rows of W accumulators, a maximum and a sum (0: not split; more than
    there are where grouped heads share row tiles)."""
    p = build_params(q, k, v, torch.empty_like(q), causal, None, None, lens, align, table)
    W = next(w for w in ((64, 128) if q.dtype == torch.float32 else (32, 64, 96, 128)) if w >= q.shape[3])
    tiles = -(-q.shape[2] // (256 if W == 128 and q.shape[2] > 128 and q.dtype != torch.float32 else 128))
    return _capi.lib().ttsdpa_workspace_bytes(ctypes.byref(p)) // (-(-q.shape[2] // 32) * 32 * (W + 2) * 4) * tiles


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%dH%dk%dL%dS%dD%d-%s-p%d" % c[:8])
def test_pieces(case, causal):
    (B, Hq, Hkv, L, S, D, dtype, page, lens), more_than = case[:9], case[9] if len(case) > 9 else 0
    q, k, v = operands(L + S, B, Hq, Hkv, L, S, D, dtype)
    if lens == "spread":
        lens = [S - (S - 1) * i // max(1, B - 1) for i in range(B)]
    n = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda")
    align = "bottom-right" if causal else "top-left"
    assert pieces(q, k, v, causal, align, n) > more_than
    got = tt.sdpAttention(q, k, v, isCausal=causal, causalAlign=align, kvLens=n)
    some = slice(None) if n is None else n > 0
    assert n is None or torch.count_nonzero(got[n == 0]).item() == 0
    # rows whose sequence is shorter than the chunk: the offset of the diagonal does not go below 0
    ref = torch.cat([reference(q[b:b + 1], k[b:b + 1], v[b:b + 1], causal and ("bottom-right" if n is None or n[b] >= L else "top-left"), None,
                               None if n is None else n[b:b + 1]) for b in range(B)])
    check(got[some], ref[some], dtype)
    kp, vp, table = scatter_to_pages(k, v, page, 5)
    n = torch.full((B,), S, dtype=torch.int32, device="cuda") if n is None else n
    assert pieces(q, kp, vp, causal, align, n, table) > more_than
    check(tt.sdpAttention(q, kp, vp, isCausal=causal, causalAlign=align, kvLens=n, blockTable=table)[some], ref[some], dtype)
