"""Products on 128 x 128 tiles whose contraction is divided among workgroups (csrc/linear.hip, launch_divided, and the merge of their
sums): few tiles and a long contraction, against float64; shares of unlike length, remainders of the tiles and of groups of four
columns, a bias, contraction-major operands (copies and sums in one scratch), and callers with less scratch."""
import ctypes

import pytest
import torch

import tinytorch_amd as tt
from tinytorch_amd import _capi

pytestmark = pytest.mark.gpu

DT = {"f32": (torch.float32, 0), "f16": (torch.float16, 1), "bf16": (torch.bfloat16, 2)}
_EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _close(got, a, b, extra=None):
    """got = a . b (+ extra): one rounding of the result and fp32 sums of K products, whose error grows at most with the sum of
    their magnitudes (K * 2^-24 of it is never reached: sqrt(K) steps of random sign, times eight)."""
    a, b = a.double(), b.double()
    ref, mag = a @ b, a.abs() @ b.abs()
    if extra is not None:
        ref, mag = ref + extra.double(), mag + extra.double().abs()
    bound = _EPS[got.dtype] * ref.abs() + 8 * a.shape[1] ** 0.5 * 2.0 ** -24 * mag + 1e-30
    worst = ((got.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, worst


def _operands(M, N, K, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + M + N + K)
    return [torch.randn(*s, generator=g, device="cuda").to(DT[dtype][0]) for s in ((M, K), (N, K), (N,))]


# tiles 24 to 112 in all, 2 to 10 shares; 103, 74 and 81 k-steps, which no number of shares here divides evenly
SIZES = [("f16", 288, 2048, 6592), ("bf16", 720, 1536, 4736), ("bf16", 129, 4097, 10368), ("bf16", 200, 4094, 14336), ("f32", 119, 3072, 9152),
         ("f32", 300, 1021, 3200), ("f16", 500, 2050, 5632), ("bf16", 978, 1024, 2688)]


@pytest.mark.parametrize("dtype,M,N,K", SIZES)
def test_divided(dtype, M, N, K):
    print("divided", dtype, M, N, K, flush=True)
    x, w, b = _operands(M, N, K, dtype)
    _close(tt.linear(x, w, b), x, w.t(), b)
    assert torch.equal(tt.linear(x, w, b), tt.linear(x, w, b))  # shares are added in one order


@pytest.mark.parametrize("dtype,M,N,K", [("bf16", 407, 17920, 3072), ("f16", 574, 13824, 2048), ("bf16", 954, 10368, 1536)])
def test_input_gradient(dtype, M, N, K):
    """grad . w with w contraction-major: the copy of w lies in the scratch before the sums."""
    print("gradient", dtype, M, N, K, flush=True)
    x, w, _ = _operands(M, N, K, dtype)
    go = _operands(M, N, N, dtype, 1)[0]
    gx, gw, gb = tt.linearBackward(go, x, w)
    _close(gx, go, w)
    _close(gw, go.t(), x)
    _close(gb.view(1, N), torch.ones(1, M, device="cuda"), go)


@pytest.mark.parametrize("dtype,M,N,K", [("bf16", 720, 1536, 4736), ("f32", 119, 3072, 9152)])
def test_less_scratch(dtype, M, N, K):
    """A caller with less than the sums need gets the same product another way; what lies behind its scratch stays as it was."""
    x, w, b = _operands(M, N, K, dtype)
    code = DT[dtype][1]
    L = _capi.lib()
    L.ttlinear_matmul_workspace_bytes.restype = ctypes.c_size_t
    i64 = ctypes.c_int64
    need = L.ttlinear_matmul_workspace_bytes(code, i64(M), i64(N), i64(K), 0, 1)
    assert need >= 2 * M * N * 4
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for size in (need, need - 256, need // 3, 0):
        ws = torch.full((need + 1024,), 77, dtype=torch.uint8, device="cuda")
        out = torch.empty(M, N, dtype=x.dtype, device="cuda")
        rc = L.ttlinear_matmul(code, p(x), p(w), p(b), p(out), i64(M), i64(N), i64(K), 0, 1, i64(K), i64(K), i64(N), p(ws), ctypes.c_size_t(size),
                               stream)
        assert rc == 0
        _close(out, x, w.t(), b)
        assert (ws[size:] == 77).all()


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(256, 4096, 2048), (257, 4096, 2048), (448, 4672, 1537), (512, 4096, 1536), (513, 4096, 1536), (220, 4608, 3072),
                                   (865, 1024, 3328), (64, 16448, 1600)])
def test_rounds_of_64_rows(dtype, M, N, K):
    """Both sides of 256 and 512 tiles of 64 x 64, where the streaming kernel's estimate counts in whole rounds."""
    print("rounds", dtype, M, N, K, flush=True)
    x, w, b = _operands(M, N, K, dtype)
    _close(tt.linear(x, w, b), x, w.t(), b)
