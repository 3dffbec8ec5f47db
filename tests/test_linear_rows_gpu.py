"""Few rows against a weight of 8192 to 16384 rows, on tiles whose two sides differ, and very large weights (csrc/linear_stream.hip,
few_rows_tile), against float64: sizes where the tile changes, remainders of it, contractions that no unit divides, unaligned rows."""
import ctypes

import pytest
import torch

import tinytorch_amd as tt
from gpu_util import CODE, close_product
from tinytorch_amd import _capi

pytestmark = pytest.mark.gpu

@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,tile", [
    (1, 8193, 64, (32, 48)), (1, 12288, 1535, (32, 48)), (16, 12289, 1000, (32, 32)), (17, 8200, 1024, (32, 48)), (32, 12288, 2048, (32, 48)),
    (31, 12287, 129, (32, 48)), (32, 12289, 1024, (32, 32)), (1, 8193, 1536, (16, 64)), (16, 16384, 2048, (16, 64)), (7, 16383, 2560, (32, 32)),
    (16, 10001, 1601, (16, 64)), (1, 8448, 2561, (32, 48)), (16, 16384, 4096, (16, 64)), (33, 9000, 512, (64, 64)), (1, 28672, 4096, (16, 16)),
    (8, 25000, 4001, (16, 16)), (5, 11000, 4096, (16, 16)), (9, 12290, 2111, (16, 64))])
def test_few_rows(M, N, K, tile, dtype):
    print("rows", M, N, K, dtype, flush=True)
    assert _capi.linear_kernel(CODE[dtype], M, N, K) == ("stream", tile, 1, 1)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w, b = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((M, K), (N, K), (N,)))
    close_product(tt.linear(x, w, b), x, w.t(), b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,tile", [
    (1, 4100, 2048, (16, 16)), (16, 8192, 2048, (16, 32)), (5, 8191, 1001, (32, 32)), (17, 8193, 1024, (32, 64)), (32, 11264, 2048, (32, 64)),
    (31, 16384, 1000, (32, 64)), (20, 16385, 1024, (32, 32)), (33, 11200, 4096, (48, 64)), (48, 17281, 3000, (48, 64)), (40, 11201, 4095, (48, 64)),
    (49, 11200, 4096, (64, 64)), (9, 6001, 1203, (16, 32)), (8, 5179, 3064, (32, 32))])
def test_few_rows_contraction_major(M, N, K, tile, dtype):
    print("rows, k-major", M, N, K, dtype, flush=True)
    assert _capi.linear_kernel(CODE[dtype], M, N, K, 0, 0) == ("stream", tile, 1, 1)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w, b = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((M, K), (K, N), (N,)))
    close_product(tt.matmul(x, w, False, False, b), x, w, b)


def test_views():
    """Rows that begin at odd elements."""
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(24, 1031, generator=g, device="cuda").half()[:, 3:]
    w = torch.randn(9001, 1033, generator=g, device="cuda").half()[:, 5:]
    b = torch.randn(9001, generator=g, device="cuda").half()
    close_product(tt.matmul(x, w, False, True, b), x, w.t(), b)
    close_product(tt.matmul(x[:5], w, False, True, b), x[:5], w.t(), b)


@pytest.mark.parametrize("M,N,K,trans_b", [(24, 9001, 1024, 1), (5, 9001, 2048, 1), (2, 28001, 4096, 1), (16, 8191, 2048, 0), (20, 9001, 1024, 0), (40, 11201, 1024, 0)])
def test_longer_rows_of_the_output(M, N, K, trans_b):
    """An output whose rows are longer than the product's, at an odd element: what lies between them stays as it was."""
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w, b = (torch.randn(*s, generator=g, device="cuda").half() for s in ((M, K), (N, K) if trans_b else (K, N), (N,)))
    for first, ldo in ((0, N + 7), (1, N + 6)):
        room = torch.full((M * ldo + 8,), 5.0, device="cuda", dtype=torch.float16)
        i64, p = ctypes.c_int64, lambda t: ctypes.c_void_p(t.data_ptr())
        rc = _capi.lib().ttlinear_matmul(_capi.F16, p(x), p(w), p(b), ctypes.c_void_p(room.data_ptr() + 2 * first), i64(M), i64(N), i64(K), 0, trans_b, i64(K),
                                         i64(w.shape[1]), i64(ldo), None, ctypes.c_size_t(0), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        out = room[first:first + M * ldo].view(M, ldo)
        close_product(out[:, :N], x, w.t() if trans_b else w, b)
        assert (out[:, N:] == 5).all() and (room[:first] == 5).all() and (room[first + M * ldo:] == 5).all()
