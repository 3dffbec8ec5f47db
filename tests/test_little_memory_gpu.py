"""Calls on a device without room for their scratch: those that can do without it run all the same, on the kernels that read their
operands in place; a call that cannot says so."""
import ctypes
import math

import pytest
import torch

import tinytorch_amd as tt
from tinytorch_amd import _capi, function

pytestmark = pytest.mark.gpu

MB = 1 << 20


class room:
    """Lets the process take `extra` bytes more device memory than it has."""

    def __init__(self, extra):
        self.extra = extra

    def __enter__(self):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + self.extra) / total)

    def __exit__(self, *exc):
        torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.fixture(params=["native", "python"])
def way(request, monkeypatch):
    if request.param == "python":
        monkeypatch.setattr(function, "_native", type("Nothing", (), {"__getattr__": lambda self, name: lambda *args: None})())
    return request.param


def rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


def operands(*shapes, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(1)
    return [torch.randn(*s, generator=g, device="cuda").to(dtype) for s in shapes]


# two bf16 results of one product: each rounded once (2^-9 at most, 2^-8 between them)
REL = 2 ** -8


def test_products(way):
    M, N, K = 4096, 4096, 4097  # an odd contraction: copies of both operands, 64 MB
    x, w = operands((M, K), (N, K))
    assert _capi.lib().ttlinear_matmul_workspace_bytes(_capi.BF16, M, N, K, 0, 1) > 60 * MB
    ref = x.float() @ w.float().t()
    with room(M * N * 2 + 8 * MB):
        y = tt.linear(x, w)
    assert rel(y, ref) <= REL
    del y
    with room(M * N * 2 + 8 * MB):
        z = tt.matmul(x, w, False, True)
    assert rel(z, ref) <= REL


def test_linear_backward(way):
    M, N, K = 2047, 2047, 2047
    x, w, g = operands((M, K), (N, K), (M, N))
    refs = (g.float() @ w.float(), g.float().t() @ x.float(), g.float().sum(0))
    torch.cuda.synchronize()
    with room(3 * M * N * 2 + M * N * 4 + 12 * MB):  # the results, and the column sums' fp32 copy
        assert _capi.lib().ttlinear_backward_workspace_bytes(_capi.BF16, M, N, K) > 8 * MB
        got = tt.linearBackward(g, x, w)
    for a, b in zip(got, refs):
        assert rel(a, b) <= REL


def test_linear_backward_in_place():
    """The weight's gradient is made on copies of its operands (75 MB): without room for them on operands as they lie.  Nor is there
    room for what the call would be made of otherwise, an fp32 copy of grad."""
    M, N, K = 2048, 9216, 4096
    x, w, g = operands((M, K), (N, K), (M, N))
    refs = (g.float() @ w.float(), g.float().t() @ x.float(), g.float().sum(0))
    L = _capi.lib()
    need, least = L.ttlinear_backward_workspace_bytes(_capi.BF16, M, N, K), L.ttlinear_backward_least_workspace_bytes(_capi.BF16, M, N)
    assert need > 60 * MB and least < MB
    torch.cuda.synchronize()
    with room((M * K + N * K) * 2 + 16 * MB):
        got = tt.linearBackward(g, x, w)
    for a, b in zip(got, refs):
        assert rel(a, b) <= REL
    # any scratch between the two is enough
    for nbytes in (least, need - 1):
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        out = [torch.empty_like(t) for t in got]
        rc = L.ttlinear_backward(_capi.BF16, g.data_ptr(), x.data_ptr(), w.data_ptr(), *[t.data_ptr() for t in out], M, N, K, N, K, K,
                                 ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert rc == 0
        for a, b in zip(out, refs):
            assert rel(a, b) <= REL


@pytest.mark.parametrize("M,N,K,dtype", [(64, 500, 784, torch.float32), (1501, 1999, 2501, torch.float32), (300, 260, 4100, torch.bfloat16),
                                         (4100, 65, 70, torch.float16)])
def test_linear_backward_with_the_least(M, N, K, dtype):
    """Products on the streaming kernel, of which the weight's would be divided, or made in one launch with the other."""
    x, w, g = operands((M, K), (N, K), (M, N), dtype=dtype)
    L = _capi.lib()
    kind = {torch.float32: _capi.F32, torch.float16: _capi.F16, torch.bfloat16: _capi.BF16}[dtype]
    least = L.ttlinear_backward_least_workspace_bytes(kind, M, N)
    assert 0 < least <= L.ttlinear_backward_workspace_bytes(kind, M, N, K)
    ws = torch.full((least + 4096,), 77, dtype=torch.uint8, device="cuda")
    out = [torch.empty(s, dtype=dtype, device="cuda") for s in ((M, K), (N, K), (N,))]
    rc = L.ttlinear_backward(kind, g.data_ptr(), x.data_ptr(), w.data_ptr(), *[t.data_ptr() for t in out], M, N, K, N, K, K, ws.data_ptr(),
                             least, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0
    assert bool((ws[least:] == 77).all())
    for a, b in zip(out, (g.double() @ w.double(), g.double().t() @ x.double(), g.double().sum(0))):
        assert rel(a, b) <= (1e-5 if dtype == torch.float32 else REL)


def test_attention(way):
    B, H, L, S, D = 1, 16, 100, 8191, 128
    q, k, v = operands((B, H, L, D), (B, H, S, D), (B, H, S, D))
    mask = torch.ones(L, S, dtype=torch.bool, device="cuda")
    mask[:, 7::9] = False
    refs = []
    for m in (None, mask):
        s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) / math.sqrt(D)
        refs.append(torch.matmul(torch.softmax(s if m is None else s.masked_fill(~m, -math.inf), -1), v.float()))
    out = torch.empty_like(q)
    for m, ref in zip((None, mask), refs):
        p = function.build_params(q, k, v, out, False, m)
        assert _capi.lib().ttsdpa_workspace_bytes(ctypes.byref(p)) > 4 * MB
        with room(2 * MB + 2 * MB):
            got = tt.sdpAttention(q, k, v, attnMask=m)
        assert rel(got, ref) <= 8e-3


def test_a_call_that_needs_it(way):
    """The decode kernels keep their partial results in scratch: without it the call names what is missing."""
    q, k, v = operands((8, 64, 1, 128), (8, 8, 4096, 128), (8, 8, 4096, 128))
    p = function.build_params(q, k, v, torch.empty_like(q))
    need = _capi.lib().ttsdpa_workspace_bytes(ctypes.byref(p))
    assert need > 2 * MB  # (not from the allocator's pool of small blocks)
    ref = tt.sdpAttention(q, k, v)
    with room(0):
        hold = []
        with pytest.raises(torch.OutOfMemoryError):
            for _ in range(64):  # what is left of larger blocks
                hold.append(torch.empty(need, dtype=torch.uint8, device="cuda"))
        with pytest.raises(torch.OutOfMemoryError):
            tt.sdpAttention(q, k, v)
    del hold
    assert torch.equal(tt.sdpAttention(q, k, v), ref)
