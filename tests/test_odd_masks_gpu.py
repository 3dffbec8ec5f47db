"""attnMasks whose rows do not begin at groups of four keys, on the matrix-core kernels: key counts around the edges of a
mask block (groups of 4, blocks of 32, tiles of 64), strided keys, and per-batch key counts beside a mask."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import TOL, backward_call, call, make_inputs, to_device, to_host_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["bool", "add"])
@pytest.mark.parametrize("dtype,D", [("f16", 64), ("bf16", 80), ("bf16", 128), ("f32", 64)])
@pytest.mark.parametrize("S", [1, 3, 5, 31, 33, 62, 65, 129, 203])
def test_odd_key_counts(S, dtype, D, kind):
    B, Hq, Hkv, L = 2, 4, 2, 37
    print("odd mask S%d %s D%d %s" % (S, dtype, D, kind), flush=True)
    host, dev = make_inputs(8800 + S, B, Hq, Hkv, L, S, D, dtype)
    rng = np.random.default_rng(S)
    if kind == "bool":
        m = rng.random((B, 1, L, S)) > 0.4
        m[..., S // 2] = True
        mh, md = m.astype(np.uint8), torch.from_numpy(m).cuda()
    else:
        mh, bits = oracle.round_to(rng.standard_normal((Hq, L, S)).astype(np.float32), dtype)
        md = to_device(mh, bits, dtype)
    rc, out = call("forward", *dev, mask=md)
    assert rc == 0
    assert np.abs(to_host_f32(out) - oracle.sdpa_f32(*host, mask=mh)).max() <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_strided_mask_and_key_counts(dtype):
    B, Hq, Hkv, L, S, D = 3, 4, 4, 70, 77, 64
    print("strided mask, key counts %s" % dtype, flush=True)
    host, dev = make_inputs(8900, B, Hq, Hkv, L, S, D, dtype)
    m = np.random.default_rng(5).random((S, L)) > 0.3
    m[0] = True
    md = torch.from_numpy(m).cuda().t()  # keys strided by L
    lens = [77, 34, 1]
    kv = torch.tensor(lens, dtype=torch.int32, device="cuda")
    rc, out = call("forward", *dev, mask=md, kv_lens=kv)
    assert rc == 0
    for b, n in enumerate(lens):
        exp = oracle.sdpa_f32(host[0][b:b + 1], host[1][b:b + 1, :, :n], host[2][b:b + 1, :, :n],
                              mask=np.ascontiguousarray(m.T[:, :n]).astype(np.uint8))
        assert np.abs(to_host_f32(out[b:b + 1]) - exp).max() <= TOL[dtype], b


def _against_64_bits(out, host, mask):
    """Relative error (2-norm), and the share of results that are not the 64-bit result rounded once."""
    q, k, v = (torch.from_numpy(t).double().cuda() for t in host)
    G = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(G, 1), v.repeat_interleave(G, 1)
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / q.shape[-1] ** 0.5
    s = s.masked_fill(~mask, -float("inf")) if mask.dtype == torch.bool else s + mask.double()
    ref = torch.matmul(torch.softmax(s, -1), v)
    return ((out.double() - ref).norm() / ref.norm()).item(), (out != ref.to(out.dtype)).double().mean().item()


@pytest.mark.parametrize("kind", ["bool", "add"])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("L,S,D", [(37, 197, 64), (197, 197, 64), (130, 333, 32), (101, 901, 80), (70, 333, 128), (33, 335, 96), (37, 203, 192),
                                   (64, 333, 256)])
@pytest.mark.parametrize("steep", [False, True])
def test_probabilities_are_fp32(L, S, D, dtype, kind, steep):
    """16-bit calls of the general route: as close to the 64-bit result as the vector-ALU kernel, whose probabilities are fp32
    (16-bit ones leave four results of ten off by a rounding).  steep: scores spread over some 20, and the key
    with the most weight holds zeros, so that the result is that of the small probabilities."""
    B, Hq, Hkv = 2, 4, 2
    print("fp32 probabilities", L, S, D, dtype, kind, steep, flush=True)
    host, dev = make_inputs(8950 + S, B, Hq, Hkv, L, S, D, dtype, 2.0 if steep else 1.0)
    rng = np.random.default_rng(S)
    m = rng.random((L, S)) > 0.3
    m[:, S // 2] = True
    md = torch.from_numpy(m).cuda()
    if kind == "add":
        md = torch.from_numpy(rng.standard_normal((L, S)).astype(np.float32)).cuda().to(dev[0].dtype)
    if steep:
        md = md.clone()
        md[:, 3] = True if kind == "bool" else 12.0
        host[2][:, :, 3] = 0
        dev[2][:, :, 3] = 0
    got, vec = call("forward", *dev, mask=md), call("general", *dev, mask=md)
    assert got[0] == 0 and vec[0] == 0
    err, off = _against_64_bits(got[1], host, md)
    err0, off0 = _against_64_bits(vec[1], host, md)
    # sums of S fp32 terms in another order: 2^-24 sqrt(S) against a rounding of 2^-12 (fp16) at most changes the result's rounding once in 2^-12 / that
    assert err <= err0 * 1.001 and off <= off0 * 1.1 + 2e-3, (err, err0, off, off0)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("S", [197, 901])
def test_infinite_values(S, dtype):
    """Infinities and NaN in V (the last key's row among them) come out where the vector-ALU kernel has them."""
    host, dev = make_inputs(8990, 2, 4, 4, 37, S, 64, dtype)
    q, k, v = dev
    m = torch.from_numpy(np.random.default_rng(1).random((37, S)) > 0.3).cuda()
    m[:, [5, 70, S - 1]] = True
    v[0, 0, 5, 3], v[0, 1, S - 1, 4], v[1, 0, 70, 7], v[1, 2, 5, :] = float("inf"), -float("inf"), float("nan"), 60000.0
    got, vec = call("forward", q, k, v, mask=m), call("general", q, k, v, mask=m)
    assert got[0] == 0 and vec[0] == 0
    assert torch.equal(got[1].isnan(), vec[1].isnan()) and torch.equal(got[1].isinf(), vec[1].isinf())
    assert torch.isinf(got[1]).any() and torch.equal(torch.sign(got[1][got[1].isinf()]), torch.sign(vec[1][vec[1].isinf()]))


def _gradients_64(host, go, md):
    q, k, v = (torch.from_numpy(t).double().cuda() for t in host)
    G, g = q.shape[1] // k.shape[1], go.double()
    kk, vv = k.repeat_interleave(G, 1), v.repeat_interleave(G, 1)
    s = torch.matmul(q, kk.transpose(-1, -2).contiguous()) / q.shape[-1] ** 0.5
    p = torch.softmax(s.masked_fill(~md, -float("inf")) if md.dtype == torch.bool else s + md.double(), -1)
    return p, q, kk, vv, g, (lambda t: t.view(t.shape[0], -1, G, *t.shape[2:]).sum(2))


@pytest.mark.parametrize("kind", ["bool", "add"])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,D", [(2, 4, 2, 37, 197, 64), (1, 1, 1, 33, 65, 32), (4, 16, 16, 260, 333, 64), (1, 4, 2, 130, 901, 80),
                                            (1, 4, 1, 70, 333, 128), (4, 16, 8, 140, 203, 120)])
@pytest.mark.parametrize("size", [1.0, 1e-6, 3e3])
def test_gradients_are_fp32(B, Hq, Hkv, L, S, D, dtype, kind, size):
    """16-bit calls of the general route: P and dS are fp32, so that an upstream gradient of any size of the type gives the 64-bit
    result rounded once (16-bit dS: off by several roundings, lost to zero below 1e-7 in fp16 and infinite beyond 65504)."""
    print("fp32 gradients", B, Hq, Hkv, L, S, D, dtype, kind, size, flush=True)
    host, dev = make_inputs(8970 + S, B, Hq, Hkv, L, S, D, dtype)
    rng = np.random.default_rng(S)
    m = rng.random((L, S)) > 0.3
    m[:, S // 2] = True
    md = torch.from_numpy(m).cuda() if kind == "bool" else torch.from_numpy(rng.standard_normal((L, S)).astype(np.float32)).cuda().to(dev[0].dtype)
    go = (torch.from_numpy(rng.standard_normal((B, Hq, L, D)).astype(np.float32)).cuda() * size).to(dev[0].dtype)
    rc, out = call("forward", *dev, mask=md)
    assert rc == 0
    rc, grads = backward_call(*dev, out, go, mask=md)
    assert rc == 0
    p, q, kk, vv, g, group = _gradients_64(host, go, md)
    # delta is dout . out with the forward's rounded output, as the backward is defined
    ds = p * (torch.matmul(g, vv.transpose(-1, -2).contiguous()) - (g * out.double()).sum(-1, keepdim=True)) / D ** 0.5
    refs = (torch.matmul(ds, kk), group(torch.matmul(ds.transpose(-1, -2).contiguous(), q)), group(torch.matmul(p.transpose(-1, -2).contiguous(), g)))
    for name, got, ref in zip(("dq", "dk", "dv"), grads, refs):
        assert torch.isfinite(got).all(), name
        # one rounding of the result, and sums of fp32 terms in another order: a rounding in a hundred may go the other way
        want = ref.to(got.dtype)
        assert (got != want).double().mean().item() <= 0.01, name
        assert ((got.double() - ref).norm() / ref.norm()).item() <= 1.001 * ((want.double() - ref).norm() / ref.norm()).item() + 1e-7, name


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("D", [64, 72, 128])
@pytest.mark.parametrize("form", ["keys strided", "per head", "per entry and key"])
def test_layouts(form, D, dtype):
    """Views of one packed buffer, masks whose keys are strided or whose rows or heads are broadcast, grouped heads: output and gradients."""
    B, Hq, Hkv, L, S = 2, 6, 2, 61, 147
    print("layouts", form, D, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(21)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[dtype])
    q = r(B, L, Hq, D + 8)[..., :D].transpose(1, 2)  # rows of wider rows, sequence outside the heads
    kv = r(B, S, 2 * Hkv, D).transpose(1, 2)
    k, v = kv[:, :Hkv], kv[:, Hkv:]
    go = r(B, L, Hq, D).transpose(1, 2)
    if form == "keys strided":
        mask = (torch.rand(S, L, generator=g, device="cuda") < 0.7).t()
        mask[:, 5] = True
    elif form == "per head":
        mask = r(Hq, 1, S)
    else:
        mask = r(B, 1, 1, 2 * S)[..., ::2]
    rc, out = call("forward", q, k, v, mask=mask)
    assert rc == 0
    rc, grads = backward_call(q, k, v, out, go, mask=mask)
    assert rc == 0
    host = [t.float().cpu().numpy() for t in (q, k, v)]
    p, qd, kk, vv, gd, group = _gradients_64(host, go, mask)
    ref = torch.matmul(p, vv)
    ds = p * (torch.matmul(gd, vv.transpose(-1, -2).contiguous()) - (gd * out.double()).sum(-1, keepdim=True)) / D ** 0.5
    refs = (ref, torch.matmul(ds, kk), group(torch.matmul(ds.transpose(-1, -2).contiguous(), qd)), group(torch.matmul(p.transpose(-1, -2).contiguous(), gd)))
    for name, got, want in zip(("out", "dq", "dk", "dv"), (out,) + tuple(grads), refs):
        rounded = want.to(got.dtype).double()
        # one rounding of the result (16-bit), and fp32 sums of some 150 products in another order
        assert ((got.double() - want).norm() / want.norm()).item() <= 1.01 * ((rounded - want).norm() / want.norm()).item() + 2e-6, name


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("D", [64, 80])
def test_pages(D, dtype):
    """The same call on a paged cache, the pages scattered: bit for bit the contiguous one's result."""
    B, H, L, S, page = 2, 4, 50, 256, 64
    host, (q, k, v) = make_inputs(8995, B, H, H, L, S, D, dtype)
    table = torch.tensor([[3, 0, 6, 1], [7, 2, 5, 4]], dtype=torch.int32, device="cuda")
    pools = []
    for t in (k, v):
        pool = torch.zeros(8, H, page, D, dtype=t.dtype, device="cuda")
        for b in range(B):
            for i in range(4):
                pool[table[b, i].item()] = t[b, :, page * i:page * (i + 1)]
        pools.append(pool)
    lens = torch.tensor([251, 130], dtype=torch.int32, device="cuda")
    mask = torch.from_numpy(np.random.default_rng(3).random((L, S)) > 0.4).cuda()
    mask[:, 0] = True
    whole, paged = call("forward", q, k, v, mask=mask, kv_lens=lens), call("forward", q, *pools, mask=mask, kv_lens=lens, block_table=table)
    assert whole[0] == 0 and paged[0] == 0 and torch.equal(whole[1], paged[1])
    vec = call("general", q, k, v, mask=mask, kv_lens=lens)
    assert (whole[1] != vec[1]).double().mean().item() <= 0.005  # (a rounding here and there)
