"""The kernels with dealt keys and the head_dim-128 backward pair on rows as a layer hands them over: q, k, v and gradients as views of packed
[B, L, (Hq + 2 Hkv) D] projections and [B, L, H D] outputs, with key counts per batch entry and several pieces of both kernels' streams at once.
Results of strided calls equal those of contiguous ones bit for bit (the kernels only differ in addresses), which are compared with float64."""
import pytest
import torch

from gpu_util import TORCH_DTYPE, backward_call, call
from tinytorch_amd import _capi
from tinytorch_amd.function import build_backward_params, build_params

pytestmark = pytest.mark.gpu

# Relative error (2-norm) of correct results, as in test_prefill_dealt_gpu.py and test_backward_streams_gpu.py.
FORWARD = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}
BACKWARD = {"f16": 2.0 ** -10, "bf16": 2.0 ** -7}


def packed(B, Hq, Hkv, L, S, D, dtype, filled=None):
    """q [B, Hq, L, D], k and v [B, Hkv, S, D]: views of a projection's rows (of two, where queries and keys differ in number), the columns
    between them filled with NaN."""
    g = torch.Generator(device="cuda").manual_seed(L + S + D)
    n = max(L, S)
    rows = torch.full((B, n, (Hq + 2 * Hkv) * D + 24), float("nan"), dtype=TORCH_DTYPE[dtype], device="cuda")
    parts = []
    for first, heads, count in ((0, Hq, L), (Hq * D + 8, Hkv, S), ((Hq + Hkv) * D + 16, Hkv, S)):
        view = rows[:, :count, first:first + heads * D].view(B, count, heads, D).transpose(1, 2)
        if filled is None:
            view.copy_(torch.randn(B, heads, count, D, device="cuda", generator=g))
        else:
            view.fill_(filled)
        parts.append(view)
    return rows, parts


def reference(q, k, v, go, causal, lens):
    """Output and gradients in 64 bits; bottom-right alignment."""
    B, Hq, L, D = q.shape
    G, dev = Hq // k.shape[1], q.device
    out, dq = (torch.zeros(q.shape, dtype=torch.float64, device=dev) for _ in range(2))
    dk, dv = (torch.zeros(k.shape, dtype=torch.float64, device=dev) for _ in range(2))
    for b, n in enumerate(lens):
        for h in range(Hq if n else 0):
            qd, kd, vd, gd = q[b, h].double(), k[b, h // G, :n].double(), v[b, h // G, :n].double(), go[b, h].double()
            s = qd @ kd.t().contiguous() / D ** 0.5
            if causal:
                s = s.masked_fill(torch.arange(n, device=dev)[None] > torch.arange(L, device=dev)[:, None] + max(0, n - L), float("-inf"))
            p = torch.softmax(s, -1)
            out[b, h] = p @ vd
            dp = gd @ vd.t().contiguous()
            ds = p * (dp - (p * dp).sum(-1, keepdim=True)) / D ** 0.5
            dq[b, h] = ds @ kd
            dk[b, h // G, :n] += ds.t().contiguous() @ qd
            dv[b, h // G, :n] += p.t().contiguous() @ gd
    return out, dq, dk, dv


def close(x, ref, rel, what):
    err = ((x.double() - ref).norm() / ref.norm()).item()
    assert err <= rel, (what, err)


@pytest.mark.parametrize("D,dtype", [(128, "bf16"), (64, "f16")])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,causal,lens,divided", [
    (1, 16, 4, 700, 700, True, None, False),
    (4, 8, 8, 514, 545, True, [545, 1, 0, 33], False),
    (4, 8, 8, 514, 545, False, [33, 545, 64, 0], False),
    (1, 4, 2, 1100, 3000, True, None, True),
])
def test_dealt_keys(B, Hq, Hkv, L, S, causal, lens, divided, D, dtype):
    _, (q, k, v) = packed(B, Hq, Hkv, L, S, D, dtype)
    rows = torch.full((B, L, Hq * D + 8), 7.0, dtype=q.dtype, device="cuda")
    out = rows[:, :, :Hq * D].view(B, L, Hq, D).transpose(1, 2)
    kv = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda")
    p = build_params(q, k, v, out, causal, None, None, kv, "bottom-right")
    assert _capi.kernel(p) == "dealt" and (_capi.division(p)[0] > 1) == divided
    rc, _ = call("forward", q, k, v, causal=causal, out=out, kv_lens=kv, align="bottom-right")
    assert rc == 0
    rc, plain = call("forward", q.contiguous(), k.contiguous(), v.contiguous(), causal=causal, kv_lens=kv, align="bottom-right")
    assert rc == 0
    assert torch.equal(out, plain) and (rows[:, :, Hq * D:] == 7.0).all()
    close(out, reference(q, k, v, torch.zeros_like(q), causal, lens or [S] * B)[0], FORWARD[dtype], "out")


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,causal,lens,pieces", [
    # are the query streams, the key ranges in several pieces?
    (1, 8, 2, 1025, 1057, True, None, (True, True)),
    (2, 8, 2, 700, 1500, False, [1500, 801], (True, True)),
    (3, 4, 2, 600, 1230, True, [1230, 0, 333], (True, True)),
    (2, 2, 1, 129, 2111, False, [2111, 1], (False, True)),
])
def test_backward_pair_in_pieces(B, Hq, Hkv, L, S, causal, lens, pieces, dtype):
    D = 128
    _, (q, k, v) = packed(B, Hq, Hkv, L, S, D, dtype)
    go = torch.randn(B, L, Hq, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)).to(q.dtype).transpose(1, 2)
    kv = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda")
    rc, out = call("forward", q, k, v, causal=causal, kv_lens=kv, align="bottom-right")
    assert rc == 0
    rows, grads = packed(B, Hq, Hkv, L, S, D, dtype, filled=7.0)
    bp = build_backward_params(q, k, v, out, go, *grads, causal, None, None, kv, "bottom-right")
    assert _capi.backward_kernel(bp) == "other" and tuple(n > 1 for n in _capi.backward_division(bp)) == pieces
    rc, _ = backward_call(q, k, v, out, go, causal, None, None, kv, "bottom-right", grads)
    assert rc == 0
    rc, plain = backward_call(q.contiguous(), k.contiguous(), v.contiguous(), out, go.contiguous(), causal, None, None, kv, "bottom-right",
                              [torch.empty_like(t, memory_format=torch.contiguous_format) for t in (q, k, v)])
    assert rc == 0
    ref = reference(q, k, v, go, causal, lens or [S] * B)
    for name, x, y, r in zip(("dq", "dk", "dv"), grads, plain, ref[1:]):
        assert torch.equal(x, y), name
        close(x, r, BACKWARD[dtype], name)
    gaps = rows.clone()
    for first, heads in ((0, Hq), (Hq * D + 8, Hkv), ((Hq + Hkv) * D + 16, Hkv)):
        gaps[:, :, first:first + heads * D] = float("nan")
    assert torch.isnan(gaps).all()
