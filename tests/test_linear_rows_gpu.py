"""Few rows against a weight of 8192 to 16384 rows, on tiles whose two sides differ, and very large weights (csrc/linear_stream.hip,
few_rows_tile), against float64: sizes where the tile changes, remainders of it, contractions that no unit divides, unaligned rows."""
import pytest
import torch

import tinytorch_amd as tt

pytestmark = pytest.mark.gpu

_EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _close(got, a, b, extra):
    """got = a . b + extra: one rounding of the result and fp32 sums of K products, whose error grows at most with the sum of their
    magnitudes (K * 2^-24 of it is never reached: sqrt(K) steps of random sign, times eight)."""
    a, b = a.double(), b.double()
    ref, mag = a @ b + extra.double(), a.abs() @ b.abs() + extra.double().abs()
    bound = _EPS[got.dtype] * ref.abs() + 8 * a.shape[1] ** 0.5 * 2.0 ** -24 * mag + 1e-30
    worst = ((got.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, worst


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [
    (1, 8193, 64), (1, 12288, 1535), (16, 12289, 1000), (17, 8200, 1024), (32, 12288, 2048), (31, 12287, 129), (32, 12289, 1024),
    (1, 8193, 1536), (16, 16384, 2048), (7, 16383, 2560), (16, 10001, 1601), (1, 8448, 2561), (16, 16384, 4096), (33, 9000, 512),
    (1, 28672, 4096), (8, 25000, 4001)])
def test_few_rows(M, N, K, dtype):
    print("rows", M, N, K, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w, b = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((M, K), (N, K), (N,)))
    _close(tt.linear(x, w, b), x, w.t(), b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [
    (1, 4100, 2048), (16, 8192, 2048), (5, 8191, 1001), (17, 8193, 1024), (32, 11264, 2048), (31, 16384, 1000), (20, 16385, 1024), (33, 11200, 4096),
    (48, 17281, 3000), (40, 11201, 4095), (49, 11200, 4096)])
def test_few_rows_contraction_major(M, N, K, dtype):
    print("rows, k-major", M, N, K, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w, b = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((M, K), (K, N), (N,)))
    _close(tt.matmul(x, w, False, False, b), x, w, b)


def test_views():
    """Rows that begin at odd elements, and an output with rows longer than the product's."""
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(24, 1031, generator=g, device="cuda").half()[:, 3:]
    w = torch.randn(9001, 1033, generator=g, device="cuda").half()[:, 5:]
    b = torch.randn(9001, generator=g, device="cuda").half()
    _close(tt.matmul(x, w, False, True, b), x, w.t(), b)
    _close(tt.matmul(x[:5], w, False, True, b), x[:5], w.t(), b)
