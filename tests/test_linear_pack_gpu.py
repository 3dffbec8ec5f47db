"""Products whose operands are first copied into whole k-tiles (rows of any length or alignment, contraction-major operands), and the
tiled kernels' stores into rows of any length: forward, both gradients, the bias gradient and every pair of transpose flags
against float64."""
import pytest
import torch

import tinytorch_amd as tt

pytestmark = pytest.mark.gpu

_EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _operand(gen, rows, cols, dtype, off):
    """[rows, cols] whose rows begin `off` elements past aligned addresses."""
    base = torch.randn(rows, cols + off, generator=gen, device="cuda").to(dtype)
    return base[:, off:]


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


# around the 128 and 256 tiles, the 64 (fp32: 32) k-tile and the copies' 64 columns and 256 rows
SIZES = [(1000, 1003, 1005), (257, 2049, 2047), (513, 1985, 1153), (2300, 700, 1301), (1025, 4095, 2050), (2049, 520, 2305)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", SIZES)
def test_layer(M, K, N, dtype):
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    x, w = _operand(gen, M, K, dtype, 0), _operand(gen, N, K, dtype, 0)
    b, go = torch.randn(N, generator=gen, device="cuda").to(dtype), _operand(gen, M, N, dtype, 0)
    _close(tt.linear(x, w, b), x, w.t(), b)
    gx, gw, gb = tt.linearBackward(go, x, w)
    _close(gx, go, w)
    _close(gw, go.t(), x)
    _close(gb.view(1, N), torch.ones(1, M, device="cuda"), go)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("dtype,off", [(torch.bfloat16, 0), (torch.bfloat16, 3), (torch.float16, 1), (torch.float32, 0), (torch.float32, 1)])
def test_flags(ta, tb, dtype, off):
    M, N, K = 1030, 1157, 1217
    gen = torch.Generator(device="cuda").manual_seed(5)
    a = _operand(gen, *((K, M) if ta else (M, K)), dtype, off)
    b = _operand(gen, *((N, K) if tb else (K, N)), dtype, off)
    bias = torch.randn(N, generator=gen, device="cuda").to(dtype)
    _close(tt.matmul(a, b, ta, tb, bias), a.t() if ta else a, b.t() if tb else b, bias)


@pytest.mark.parametrize("M,K,N", [(4096, 2048, 2048), (1999, 4096, 6144)])
def test_large_tiles_with_copies(M, K, N):
    """Whole chip on 256 x 256 tiles: the copies' column sums, rows that end inside a tile, infinities kept where they belong."""
    gen = torch.Generator(device="cuda").manual_seed(9)
    dtype = torch.bfloat16
    x, w, go = _operand(gen, M, K, dtype, 0), _operand(gen, N, K, dtype, 0), _operand(gen, M, N, dtype, 0)
    gx, gw, gb = tt.linearBackward(go, x, w)
    _close(gx, go, w)
    _close(gw, go.t(), x)
    _close(gb.view(1, N), torch.ones(1, M, device="cuda"), go)
    x[M - 1, K - 1] = float("inf")
    y = tt.linear(x, w)
    assert torch.isfinite(y[:M - 1]).all() and torch.isinf(y[M - 1]).all()
