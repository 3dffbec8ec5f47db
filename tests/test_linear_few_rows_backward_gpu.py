"""Gradients of a layer over few rows, against float64: a contraction of one to eight units of the streaming kernel's tiles, whose
workgroups take as many tiles as leave no wavefront idle (csrc/linear_stream.hip, tile_wavefronts), with a last workgroup not full of
them; and large tiles of short contractions."""
import pytest
import torch

import tinytorch_amd as tt

pytestmark = pytest.mark.gpu

_EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}
_TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _close(got, a, b):
    """got = a . b: one rounding of the result and fp32 sums of K products, whose error grows at most with the sum of their
    magnitudes (K * 2^-24 of it is never reached: sqrt(K) steps of random sign, times eight).  fp16 below its normal numbers (one product
    of two small ones) is rounded to multiples of 2^-24: half of that."""
    a, b = a.double(), b.double()
    ref, mag = a @ b, a.abs() @ b.abs()
    bound = _EPS[got.dtype] * ref.abs() + 8 * a.shape[1] ** 0.5 * 2.0 ** -24 * mag + (2.0 ** -25 if got.dtype == torch.float16 else 1e-30)
    worst = ((got.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, worst


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("M", [1, 17, 32, 33, 64, 65, 100, 128, 129, 255, 257])
@pytest.mark.parametrize("N,K", [(100, 97), (500, 784), (1001, 333)])
def test_backward(dtype, M, N, K):
    print("few rows", dtype, M, N, K, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    go, x, w = (torch.randn(*s, generator=g, device="cuda").to(_TYPES[dtype]) for s in ((M, N), (M, K), (N, K)))
    gx, gw, gb = tt.linearBackward(go, x, w)
    _close(gx, go, w)
    _close(gw, go.t(), x)
    _close(gb.view(1, N), torch.ones(1, M, device="cuda"), go)


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(1, 128, 4096), (16, 2048, 2048), (17, 4001, 1111), (31, 3000, 1000), (32, 2047, 1536), (33, 2048, 2048), (64, 1023, 2049),
                                   (65, 2048, 1024), (128, 1536, 1535), (129, 3071, 257), (255, 1500, 2000), (256, 2048, 1536), (257, 2048, 1536)])
def test_large_tiles(dtype, M, N, K):
    """128 x 128 tiles of the weight's gradient (csrc/linear_outer.hip): units of the contraction and remainders of them, last tiles that
    are moved back, unaligned rows; both with the bias's gradient and through matmul with a bias."""
    test_backward(dtype, M, N, K)
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b, c = (torch.randn(*s, generator=g, device="cuda").to(_TYPES[dtype]) for s in ((M, N + 1), (M, K + 3), (K,)))
    got = tt.matmul(a[:, 1:], b[:, 3:], True, False, c)
    one = torch.ones(N, 1, device="cuda", dtype=a.dtype)
    _close(got, torch.cat((a[:, 1:].t(), one), 1), torch.cat((b[:, 3:], c.view(1, K)), 0))


@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_batch(dtype):
    """Entries of one launch with both operands contraction-major, rows at odd elements."""
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randn(5, 40, 203, generator=g, device="cuda").to(_TYPES[dtype])
    b = torch.randn(5, 40, 75, generator=g, device="cuda").to(_TYPES[dtype])
    got = tt.matmul(a, b, True, False)
    for i in range(5):
        _close(got[i], a[i].t(), b[i])
