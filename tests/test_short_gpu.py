"""Short sequences, forward and backward (csrc/sdpa_short.hip), against the chain matmul -> scale -> mask -> softmax -> matmul
(reference src/Function/FuncNNLayer.h:237-265) and its gradients in 64 bits: sizes around the kernels' units of 16 rows and keys and
their eight wavefronts, every element type, head sizes of 8 to 128, both causal alignments, key counts, grouped heads whose units are
divided among workgroups, gradients in one launch (up to about 130 rows) and in two."""
import ctypes
import math

import pytest
import torch

import tinytorch_amd as tt
from gpu_util import backward_call, call
from tinytorch_amd import _capi, build_backward_params

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# relative error of a whole result (2-norm).  16 bits: the rounding of the probabilities (or of dS and the output that delta is
# formed from) and that of the result, half a step at most each: 2 to 3 times 2^-11 or 2^-8, the mean square being a third of that.
# fp32: sums of up to 1000 products in a few chains and the hardware's exp2 and log2, some 2^-22.
REL = {"f32": 3e-6, "f16": 2 ** -11 * 1.6, "bf16": 2 ** -8 * 1.6}

CASES = [
    # B, Hq, Hkv, L, S, D, causal ("br": bottom-right aligned), key counts
    (1, 2, 2, 16, 16, 64, True, None),          # one unit
    (1, 2, 1, 17, 31, 64, False, None),
    (2, 2, 2, 31, 17, 128, True, None),         # rows past S see every key
    (1, 4, 4, 64, 64, 64, True, None),
    (1, 4, 4, 100, 100, 80, True, None),
    (1, 3, 1, 127, 129, 128, False, None),      # eight units and one key
    (1, 4, 4, 128, 128, 64, True, None),
    (2, 8, 2, 129, 129, 64, True, None),        # nine units; groups of four heads divided
    (1, 7, 1, 90, 90, 128, True, None),
    (2, 4, 2, 150, 200, 96, "br", None),
    (2, 2, 2, 200, 150, 64, "br", None),        # more rows than keys
    (3, 4, 2, 100, 160, 64, "br", (160, 77, 101)),
    (3, 2, 2, 120, 120, 128, False, (1, 120, 63)),
    (4, 2, 1, 60, 70, 64, False, (70, 0, 16, 33)),  # an entry without keys
    (1, 8, 2, 333, 333, 128, True, None),       # gradients in two launches and divided
    (2, 2, 2, 500, 511, 64, False, None),
    (1, 2, 1, 1000, 1000, 64, True, None),
    (1, 2, 2, 48, 48, 8, True, None),
    (1, 2, 2, 48, 40, 40, False, None),
    (2, 16, 16, 260, 260, 64, True, None),      # more workgroups than CUs
]


def operands(seed, B, Hq, Hkv, L, S, D, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(B, h, n, D, generator=g, device="cuda").to(DT[dtype]) for h, n in ((Hq, L), (Hkv, S), (Hkv, S), (Hq, L))]


def expected(q, k, v, go, causal, lens):
    """Output and gradients in 64 bits on the CPU; batch entries without keys: zeros."""
    q, k, v, go = (x.double().cpu().requires_grad_() for x in (q, k, v, go))
    B, Hq, L, D = q.shape
    S, G = k.shape[2], Hq // k.shape[1]
    s = torch.matmul(q, k.repeat_interleave(G, 1).transpose(-1, -2).contiguous()) / math.sqrt(D)
    n = torch.tensor(lens if lens else [S] * B)
    hidden = (torch.arange(S)[None] >= n[:, None])[:, None, None, :].expand(B, 1, L, S)
    if causal:
        off = (n - L).clamp(min=0) if causal == "br" else torch.zeros_like(n)
        hidden = hidden | (torch.arange(S)[None, None, None] > (torch.arange(L)[None, :, None] + off[:, None, None])[:, None])
    p = torch.softmax(s.masked_fill(hidden, -math.inf), -1)
    p = torch.where((n == 0)[:, None, None, None], torch.zeros_like(p), p)
    out = torch.matmul(p, v.repeat_interleave(G, 1))
    return (out.detach(),) + tuple(x.nan_to_num() for x in torch.autograd.grad(out, (q, k, v), go))


def rel_err(got, ref):
    return ((got.double().cpu() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("dtype", list(DT))
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%dH%dk%dL%dS%dD%d-%s-%s" % (c[:7] + ("all" if c[7] is None else "lens",)))
def test_short(case, dtype):
    B, Hq, Hkv, L, S, D, causal, lens = case
    print("short", case, dtype, flush=True)
    q, k, v, go = operands(L + S + D, B, Hq, Hkv, L, S, D, dtype)
    n = torch.tensor(lens, dtype=torch.int32, device="cuda") if lens else None
    kw = dict(isCausal=bool(causal), kvLens=n, causalAlign="bottom-right" if causal == "br" else "top-left")
    out = tt.sdpAttention(q, k, v, **kw)
    got = (out,) + tuple(tt.sdpAttentionBackward(go, q, k, v, out, **kw))
    for name, x, y in zip(("out", "dq", "dk", "dv"), got, expected(q, k, v, go, causal, lens)):
        assert rel_err(x, y) <= REL[dtype], (name, rel_err(x, y))
    if lens:
        for b, m in enumerate(lens):
            assert not got[2][b, :, m:].any() and not got[3][b, :, m:].any()


@pytest.mark.parametrize("dtype", list(DT))
def test_strided_views(dtype):
    """q, k and v as views of one packed projection, gradients of an output that is not dense."""
    B, L, H, D = 2, 75, 4, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    qkv = torch.randn(B, L, 3 * H, D, generator=g, device="cuda").to(DT[dtype]).transpose(1, 2)
    q, k, v = qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:]
    go = torch.randn(B, L, H, D, generator=g, device="cuda").to(DT[dtype]).transpose(1, 2)
    out = tt.sdpAttention(q, k, v, isCausal=True)
    got = (out,) + tuple(tt.sdpAttentionBackward(go, q, k, v, out, isCausal=True))
    for x, y in zip(got, expected(q, k, v, go, True, None)):
        assert rel_err(x, y) <= REL[dtype]


@pytest.mark.parametrize("dtype", list(DT))
def test_nan_reaches_the_gradients(dtype):
    """A NaN in q is a NaN row of the output and of dq, and reaches dk and dv; other rows of dq are clean."""
    q, k, v, go = operands(5, 1, 2, 2, 64, 64, 64, dtype)
    q[0, 0, 20, 3] = math.nan
    out = tt.sdpAttention(q, k, v)
    dq, dk, dv = tt.sdpAttentionBackward(go, q, k, v, out)
    assert out[0, 0, 20].isnan().all() and dq[0, 0, 20].isnan().all()
    assert dk[0, 0].isnan().any() and dv[0, 0].isnan().any()
    assert not dq[0, 0, :20].isnan().any() and not dq[0, 1].isnan().any() and not dk[0, 1].isnan().any()


@pytest.mark.parametrize("L", [128, 300])
def test_less_scratch(L):
    """A caller whose scratch holds the pairs' needs only (4 x 8 heads on 2: the divided sums of the short way need more) gets the
    same gradients; one byte of statistics less is refused."""
    q, k, v, go = operands(9, 1, 8, 2, L, L, 128, "bf16")
    out = tt.sdpAttention(q, k, v, isCausal=True)
    ref = expected(q, k, v, go, True, None)[1:]
    d = [torch.empty_like(x) for x in (q, k, v)]
    p = build_backward_params(q, k, v, out, go, *d, True, None, None, None, "top-left")
    need = _capi.lib().ttsdpa_backward_workspace_bytes(ctypes.byref(p))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ran = 0
    for size in (need, need // 2, need // 4, 8 * 8 * L - 1):
        for x in d:
            x.fill_(7)
        rc = _capi.lib().ttsdpa_backward(ctypes.byref(p), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(size), stream)
        if rc == 0:
            ran += 1
            for x, y in zip(d, ref):
                assert rel_err(x, y) <= REL["bf16"]
        else:
            assert rc == _capi.ERR_WORKSPACE
    assert ran >= 1 and rc == _capi.ERR_WORKSPACE
