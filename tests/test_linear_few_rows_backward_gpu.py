"""Gradients of a layer over few rows, against float64: a contraction of one to eight units of the streaming kernel's tiles, whose
workgroups take as many tiles as leave no wavefront idle (csrc/linear_stream.hip, waves_of_call), with a last workgroup not full of
them; and large tiles of short contractions."""
import pytest
import torch

import tinytorch_amd as tt
from gpu_util import CODE, close_product
from tinytorch_amd import _capi

pytestmark = pytest.mark.gpu

_TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("M", [1, 17, 32, 33, 64, 65, 100, 128, 129, 255, 257])
@pytest.mark.parametrize("N,K", [(100, 97), (500, 784), (1001, 333)])
def test_backward(dtype, M, N, K):
    """Both products in one launch; 1, 2, 4 or 8 tiles of the weight's gradient to a workgroup."""
    of_weight, _, one = _capi.linear_backward_kernels(CODE[_TYPES[dtype]], M, N, K)
    units = -(-M // (32 if dtype == "f32" else 64))
    assert one and of_weight[0] == "stream" and of_weight[2] == (1 if N == 100 else max(8 >> (units - 1).bit_length(), 1))
    backward(dtype, M, N, K)


def backward(dtype, M, N, K):
    print("few rows", dtype, M, N, K, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    go, x, w = (torch.randn(*s, generator=g, device="cuda").to(_TYPES[dtype]) for s in ((M, N), (M, K), (N, K)))
    gx, gw, gb = tt.linearBackward(go, x, w)
    close_product(gx, go, w)
    close_product(gw, go.t(), x)
    close_product(gb.view(1, N), torch.ones(1, M, device="cuda"), go)


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(1, 128, 4096), (16, 2048, 2048), (17, 4001, 1111), (31, 3000, 1000), (32, 2047, 1536), (33, 2048, 2048), (64, 1023, 2049),
                                   (65, 2048, 1024), (128, 1536, 1535), (129, 3071, 257), (255, 1500, 2000), (256, 2048, 1536), (257, 2048, 1536)])
def test_large_tiles(dtype, M, N, K):
    """128 x 128 tiles of the weight's gradient (csrc/linear_outer.hip): units of the contraction and remainders of them, last tiles that
    are moved back, unaligned rows; both with the bias's gradient and through matmul with a bias."""
    assert (_capi.linear_kernel(CODE[_TYPES[dtype]], N, K, M, 1, 0)[0] == "outer") == (M <= 32 if dtype == "f32" else M < 256) or M == 1
    assert dtype == "f32" or M in (1, 257) or _capi.linear_backward_kernels(CODE[_TYPES[dtype]], M, N, K)[0][0] == "outer"
    backward(dtype, M, N, K)
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b, c = (torch.randn(*s, generator=g, device="cuda").to(_TYPES[dtype]) for s in ((M, N + 1), (M, K + 3), (K,)))
    got = tt.matmul(a[:, 1:], b[:, 3:], True, False, c)
    one = torch.ones(N, 1, device="cuda", dtype=a.dtype)
    close_product(got, torch.cat((a[:, 1:].t(), one), 1), torch.cat((b[:, 3:], c.view(1, K)), 0))


@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_batch(dtype):
    """Entries of one launch with both operands contraction-major, rows at odd elements."""
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randn(5, 40, 203, generator=g, device="cuda").to(_TYPES[dtype])
    b = torch.randn(5, 40, 75, generator=g, device="cuda").to(_TYPES[dtype])
    got = tt.matmul(a, b, True, False)
    for i in range(5):
        close_product(got[i], a[i].t(), b[i])
