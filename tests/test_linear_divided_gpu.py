"""Products on 128 x 128 tiles whose contraction is divided among workgroups (csrc/linear.hip, launch_divided, and the merge of their
sums): few tiles and a long contraction, against float64; shares of unlike length, remainders of the tiles and of groups of four
columns, a bias, contraction-major operands (copies and sums in one scratch), and callers with less scratch."""
import ctypes

import pytest
import torch

import tinytorch_amd as tt
from gpu_util import close_product
from tinytorch_amd import _capi

pytestmark = pytest.mark.gpu

DT = {"f32": (torch.float32, 0), "f16": (torch.float16, 1), "bf16": (torch.bfloat16, 2)}
def _operands(M, N, K, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + M + N + K)
    return [torch.randn(*s, generator=g, device="cuda").to(DT[dtype][0]) for s in ((M, K), (N, K), (N,))]


# tiles 48 to 72 in all; 103, 74 and 81 k-steps, which no number of shares here divides evenly
SIZES = [("f16", 288, 2048, 6592, 5), ("bf16", 720, 1536, 4736, 3), ("bf16", 129, 4097, 10368, 3), ("bf16", 200, 4094, 14336, 4), ("f16", 500, 2050, 5632, 3)]


@pytest.mark.parametrize("dtype,M,N,K,shares", SIZES)
def test_divided(dtype, M, N, K, shares):
    print("divided", dtype, M, N, K, flush=True)
    assert _capi.linear_kernel(DT[dtype][1], M, N, K) == ("tiled", (0, 0), 1, shares)
    x, w, b = _operands(M, N, K, dtype)
    close_product(tt.linear(x, w, b), x, w.t(), b)
    assert torch.equal(tt.linear(x, w, b), tt.linear(x, w, b))  # shares are added in one order


@pytest.mark.parametrize("trans_b", [0, 1])
@pytest.mark.parametrize("M,N,K", [(6, 768, 28672), (15, 3000, 16385), (1, 500, 4097)])
def test_narrow_operand(M, N, K, trans_b):
    """fp32 is divided where the streaming kernel does not take it: a contraction-major operand of fewer than 16 rows, whose copy (and
    that of the other one) lies in the scratch before the sums."""
    print("narrow", M, N, K, trans_b, flush=True)
    kernel = _capi.linear_kernel(_capi.F32, M, N, K, 1, trans_b)
    assert kernel[0] == "tiled" and kernel[3] > 1
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b, c = (torch.randn(*s, generator=g, device="cuda") for s in ((K, M), (N, K) if trans_b else (K, N), (N,)))
    close_product(tt.matmul(a, b, True, bool(trans_b), c), a.t(), b.t() if trans_b else b, c)


@pytest.mark.parametrize("dtype,M,N,K,shares", [("bf16", 535, 19072, 2048, 3), ("f16", 809, 16576, 1024, 4), ("bf16", 954, 10368, 1536, 2)])
def test_input_gradient(dtype, M, N, K, shares):
    """grad . w with w contraction-major: the copy of w lies in the scratch before the sums."""
    print("gradient", dtype, M, N, K, flush=True)
    assert _capi.linear_backward_kernels(DT[dtype][1], M, N, K)[1] == ("tiled", (0, 0), 1, shares)
    x, w, _ = _operands(M, N, K, dtype)
    go = _operands(M, N, N, dtype, 1)[0]
    gx, gw, gb = tt.linearBackward(go, x, w)
    close_product(gx, go, w)
    close_product(gw, go.t(), x)
    close_product(gb.view(1, N), torch.ones(1, M, device="cuda"), go)


@pytest.mark.parametrize("dtype,M,N,K", [("bf16", 720, 1536, 4736), ("f16", 288, 2048, 6592)])
def test_less_scratch(dtype, M, N, K):
    """A caller with less than the sums need gets the same product another way; what lies behind its scratch stays as it was."""
    assert _capi.linear_kernel(DT[dtype][1], M, N, K)[0] == "tiled"
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
        close_product(out, x, w.t(), b)
        assert (ws[size:] == 77).all()


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(256, 4096, 2048), (257, 4096, 2048), (448, 4672, 1537), (512, 4096, 1536), (513, 4096, 1536), (220, 4608, 3072),
                                   (865, 1024, 3328), (64, 16448, 1600)])
def test_rounds_of_64_rows(dtype, M, N, K):
    """Both sides of 256 and 512 tiles of 64 x 64, where the streaming kernel's estimate counts in whole rounds."""
    print("rounds", dtype, M, N, K, flush=True)
    x, w, b = _operands(M, N, K, dtype)
    close_product(tt.linear(x, w, b), x, w.t(), b)
