"""Short sequences, forward and backward (csrc/sdpa_short.hip; each case says which of its calls run there), against the chain matmul -> scale -> mask -> softmax -> matmul
(reference src/Function/FuncNNLayer.h:237-265) and its gradients in 64 bits: sizes around the kernels' units of 16 rows and keys and
their eight wavefronts, every element type, head sizes of 8 to 128, both causal alignments, key counts, grouped heads whose units are
divided among workgroups, more workgroups than CUs, gradients in one launch and in two."""
import ctypes
import math

import pytest
import torch

import tinytorch_amd as tt
from tinytorch_amd import _capi, build_backward_params
from tinytorch_amd.function import build_params

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# relative error of a whole result (2-norm).  16 bits: the rounding of the probabilities (or of dS and the output that delta is
# formed from) and that of the result, half a step at most each: 2 to 3 times 2^-11 or 2^-8, the mean square being a third of that.
# fp32: sums of up to 1000 products in a few chains and the hardware's exp2 and log2, some 2^-22.
REL = {"f32": 3e-6, "f16": 2 ** -11 * 1.6, "bf16": 2 ** -8 * 1.6}

CASES = [
    # B, Hq, Hkv, L, S, D, causal ("br": bottom-right aligned), key counts; kernels of fp32 forward and backward, 16-bit forward and
    # backward: s(hort; backward: dq, then dk and dv), j(oint: one launch), o(ther)
    (1, 2, 2, 16, 16, 64, True, None, "sjoj"),          # one unit
    (1, 2, 1, 17, 31, 64, False, None, "sjoj"),
    (2, 2, 2, 31, 17, 128, True, None, "ossj"),         # rows past S see every key
    (1, 4, 4, 64, 64, 64, True, None, "sjoj"),
    (1, 4, 4, 100, 100, 80, True, None, "sssj"),
    (1, 3, 1, 127, 129, 128, False, None, "sosj"),      # eight units and one key
    (1, 4, 4, 128, 128, 64, True, None, "sjsj"),
    (2, 8, 2, 129, 129, 64, True, None, "sjsj"),        # nine units; groups of four heads divided
    (1, 7, 1, 90, 90, 128, True, None, "sssj"),
    (2, 4, 2, 150, 200, 96, "br", None, "sosj"),
    (2, 2, 2, 200, 150, 64, "br", None, "sjsj"),        # more rows than keys
    (3, 4, 2, 100, 160, 64, "br", (160, 77, 101), "sjsj"),
    (3, 2, 2, 120, 120, 128, False, (1, 120, 63), "sssj"),
    (4, 2, 1, 60, 70, 64, False, (70, 0, 16, 33), "sjsj"),  # an entry without keys
    (1, 8, 2, 333, 333, 128, True, None, "ssss"),       # gradients in two launches and divided
    (2, 2, 2, 500, 511, 64, False, None, "soss"),
    (1, 2, 1, 1000, 1000, 64, True, None, "soss"),
    (1, 2, 2, 48, 48, 8, True, None, "sjoj"),
    (1, 2, 2, 48, 40, 40, False, None, "sjoj"),
    (2, 16, 16, 260, 260, 64, True, None, "sooo"),      # more workgroups than CUs, in each of the kernels
    (2, 8, 8, 300, 300, 64, True, None, "ooso"),
    (2, 8, 2, 333, 333, 64, True, None, "ooss"),
    (8, 8, 8, 72, 72, 64, True, None, "oooj"),
    (1, 16, 2, 330, 330, 64, True, None, "osss"),
    (1, 32, 4, 130, 130, 64, True, None, "ojoj"),
    (1, 64, 8, 70, 70, 128, True, None, "ossj"),
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
    B, Hq, Hkv, L, S, D, causal, lens, kernels = case
    print("short", case, dtype, flush=True)
    q, k, v, go = operands(L + S + D, B, Hq, Hkv, L, S, D, dtype)
    n = torch.tensor(lens, dtype=torch.int32, device="cuda") if lens else None
    kw = dict(isCausal=bool(causal), kvLens=n, causalAlign="bottom-right" if causal == "br" else "top-left")
    out = tt.sdpAttention(q, k, v, **kw)
    args = (bool(causal), None, None, n, kw["causalAlign"])
    letter = {"short": "s", "short_joint": "j", "other": "o"}
    ran = letter[_capi.kernel(build_params(q, k, v, out, *args))] + letter[_capi.backward_kernel(build_backward_params(q, k, v, out, go, q, k, v, *args))]
    assert ran == (kernels[:2] if dtype == "f32" else kernels[2:])
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


def test_less_scratch():
    """A caller whose scratch is less than the divided sums of the short way need, but enough for the kernels of long sequences, gets
    the same gradients from those; with less it is refused."""
    B, Hq, Hkv, L, S, D = 3, 4, 2, 100, 160, 64
    lens = (160, 77, 101)
    q, k, v, go = operands(9, B, Hq, Hkv, L, S, D, "bf16")
    n = torch.tensor(lens, dtype=torch.int32, device="cuda")
    out = tt.sdpAttention(q, k, v, isCausal=True, kvLens=n, causalAlign="bottom-right")
    ref = expected(q, k, v, go, "br", lens)[1:]
    d = [torch.empty_like(x) for x in (q, k, v)]
    p = build_backward_params(q, k, v, out, go, *d, True, None, None, n, "bottom-right")
    need, least = _capi.lib().ttsdpa_backward_workspace_bytes(ctypes.byref(p)), 8 * B * Hq * L
    assert need > 2 * least
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for size, kernel in ((need, "short_joint"), (need - 1, "other"), (least, "other")):
        assert _capi.backward_kernel(p, size) == kernel
        for x in d:
            x.fill_(7)
        assert _capi.lib().ttsdpa_backward(ctypes.byref(p), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(size), stream) == 0
        for x, y in zip(d, ref):
            assert rel_err(x, y) <= REL["bf16"]
    assert _capi.lib().ttsdpa_backward(ctypes.byref(p), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(least - 1), stream) == _capi.ERR_WORKSPACE
