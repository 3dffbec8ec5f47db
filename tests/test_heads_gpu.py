"""Short sequences of many heads with an attnMask (csrc/sdpa_heads.hip), against the chain matmul -> scale -> mask -> softmax -> matmul
(reference src/Function/FuncNNLayer.h:237-265) in 64 bits: sizes around the kernel's units of 16 keys, its pairs of them and its eight
wavefronts, masks of the keys alone (broadcast, strided, with holes) and with rows, key counts beside them, grouped heads, rows that see
no key, infinities in V."""
import math

import pytest
import torch

import tinytorch_amd as tt
from tinytorch_amd import _capi
from tinytorch_amd.function import build_params

pytestmark = pytest.mark.gpu

DT = {"f16": torch.float16, "bf16": torch.bfloat16}
# relative error of a whole result (2-norm): the rounding of the result, at most one half step of the type, and of probabilities
# that the call's route rounds to it
REL = {"f16": 2 ** -11 * 1.6, "bf16": 2 ** -8 * 1.6}

CASES = [
    # B, Hq, Hkv, L, S, D, mask
    (2, 4, 4, 16, 1, 64, "keys"),       # one key
    (2, 4, 4, 17, 15, 8, "keys"),
    (3, 4, 2, 31, 33, 64, "keys"),      # two pairs of units, the second of one key; grouped heads
    (2, 2, 2, 130, 97, 40, "keys"),     # nine row units: two workgroups a head
    (16, 12, 12, 197, 197, 64, "keys"),
    (2, 4, 4, 256, 256, 64, "keys"),
    (40, 8, 8, 129, 130, 64, "keys"),   # 32 rows a wavefront
    (40, 8, 8, 250, 256, 48, "keys"),
    (33, 8, 8, 16, 64, 56, "keys"),
    (3, 4, 4, 100, 100, 64, "holes"),
    (3, 4, 4, 64, 64, 64, "holes"),
    (2, 4, 4, 60, 61, 64, "strided"),
    (3, 4, 4, 70, 90, 64, "counts"),
    (40, 8, 8, 200, 200, 64, "counts"),
    (2, 4, 4, 16, 4, 64, "add"),
    (2, 4, 2, 77, 129, 64, "add"),      # contiguous keys that no group of four ends with
    (1, 4, 4, 256, 255, 64, "add"),
    (2, 4, 4, 64, 128, 24, "add"),
    (2, 4, 4, 90, 75, 64, "bool"),
    (2, 4, 4, 128, 252, 64, "bool"),
]


def make_mask(kind, B, H, L, S, g):
    dev = "cuda"
    n = torch.randint(1, S + 1, (B,), generator=g, device=dev)
    n[0] = S
    if kind in ("keys", "counts"):
        return (torch.arange(S, device=dev)[None] < n[:, None]).view(B, 1, 1, S)
    if kind == "holes":
        m = torch.rand(B, 1, 1, S, generator=g, device=dev) < 0.4
        m[:, :, :, S // 2] = True
        return m
    if kind == "strided":
        m = torch.rand(B, 1, 1, 3 * S, generator=g, device=dev) < 0.5
        m[..., 0] = True
        return m[..., ::3]
    if kind == "add":
        return torch.randn(H, L, S, generator=g, device=dev)
    m = torch.rand(B, 1, L, S, generator=g, device=dev) < 0.5
    m[..., 0] = True
    return m


def expected(q, k, v, mask, lens):
    q, k, v = (x.double().cpu() for x in (q, k, v))
    G, S = q.shape[1] // k.shape[1], k.shape[2]
    s = torch.matmul(q, k.repeat_interleave(G, 1).transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    mask = mask.cpu()
    s = s.masked_fill(~mask, -math.inf) if mask.dtype == torch.bool else s + mask.double()
    if lens is not None:
        s = s.masked_fill((torch.arange(S)[None] >= lens.cpu()[:, None])[:, None, None], -math.inf)
    return torch.matmul(torch.softmax(s, -1), v.repeat_interleave(G, 1))


@pytest.mark.parametrize("dtype", list(DT))
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%dH%dk%dL%dS%dD%d-%s" % c)
def test_heads(case, dtype):
    B, Hq, Hkv, L, S, D, kind = case
    print("heads", case, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(L + S + D)
    q, k, v = (torch.randn(B, h, n, D, generator=g, device="cuda").to(DT[dtype]) for h, n in ((Hq, L), (Hkv, S), (Hkv, S)))
    mask = make_mask(kind, B, Hq, L, S, g)
    if mask.dtype != torch.bool:
        mask = mask.to(DT[dtype])
    lens = None
    if kind == "counts":  # key counts beside the mask; the first key of every entry is visible
        lens = torch.randint(1, S + 1, (B,), generator=g, device="cuda", dtype=torch.int32)
    out = tt.sdpAttention(q, k, v, attnMask=mask, kvLens=lens)
    assert _capi.kernel(build_params(q, k, v, out, False, mask, None, lens)) == ("heads_32" if B == 40 or B == 16 else "heads_16")
    ref = expected(q, k, v, mask, lens)
    err = ((out.double().cpu() - ref).norm() / ref.norm()).item()
    assert err <= REL[dtype], err


@pytest.mark.parametrize("dtype", list(DT))
@pytest.mark.parametrize("B,H,L", [(2, 4, 45), (2, 4, 64), (40, 8, 150)])
def test_rows_and_values_at_the_edge(B, H, L, dtype):
    """Batch entries whose keys are all hidden: NaN.  A NaN in a hidden key's k: nothing.  An infinity in v: its column alone, in
    every row that gives the key weight; NaN there where the key is hidden (0 times it, as in the reference's chain)."""
    D = 64
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(B, H, L, D, generator=g, device="cuda").to(DT[dtype]) for _ in "qkv")
    mask = make_mask("keys", B, H, L, L, g)
    mask[1] = False
    mask[0, :, :, L - 3:] = False
    k[0, 0, L - 1] = math.nan
    out = tt.sdpAttention(q, k, v, attnMask=mask)
    assert _capi.kernel(build_params(q, k, v, out, False, mask)) == ("heads_32" if B == 40 else "heads_16")
    ref = expected(q, k.nan_to_num(), v, mask, None)
    assert out[1].isnan().all()
    seen = torch.ones(B, dtype=torch.bool)
    seen[1] = False
    seen &= mask.view(B, L).any(1).cpu()
    assert ((out.double().cpu()[seen] - ref[seen]).norm() / ref[seen].norm()).item() <= REL[dtype]
    v[0, 1, 2, 5] = math.inf      # visible
    v[0, 2, L - 2, 7] = math.inf  # hidden
    out2 = tt.sdpAttention(q, k, v, attnMask=mask)
    assert (out2[0, 1, :, 5] == math.inf).all() and out2[0, 2, :, 7].isnan().all()
    out2[0, 1, :, 5], out2[0, 2, :, 7] = out[0, 1, :, 5], out[0, 2, :, 7]
    assert torch.equal(out2[0], out[0])


@pytest.mark.parametrize("dtype", list(DT))
def test_lowest_value(dtype):
    """Rows whose biases are all the type's lowest value: equal weights, as the reference's chain gives them."""
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn(2, 4, 50, 64, generator=g, device="cuda").to(DT[dtype]) for _ in "qkv")
    mask = torch.zeros(4, 50, 50, device="cuda", dtype=DT[dtype])
    mask[:, 7] = torch.finfo(DT[dtype]).min
    out = tt.sdpAttention(q, k, v, attnMask=mask)
    assert _capi.kernel(build_params(q, k, v, out, False, mask)) == "heads_16"
    assert out.isfinite().all()
    if dtype == "bf16":  # (fp16's lowest value leaves the scores their bits)
        mean = v.double().mean(2)
        assert ((out[:, :, 7].double() - mean).norm() / mean.norm()).item() <= REL[dtype]
