"""softmax / logSoftmax and their backwards over rows of every kind of length: below one 16-byte vector, odd lengths whose rows
begin at any element, the boundaries between the kernels' row shapes, rows longer than a workgroup keeps in registers;
tensors that lie differently from each other; results written over the input.  Against the same formulas in float64."""
import numpy as np
import pytest
import torch

from gpu_util import TORCH_DTYPE
from tinytorch_amd import _capi

pytestmark = pytest.mark.gpu

CODE = {"f32": _capi.F32, "f16": _capi.F16, "bf16": _capi.BF16}
EPS = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}  # half a unit in the last place


def placed(t, shift):
    """A copy of t that begins `shift` elements into a buffer."""
    buf = torch.zeros(t.numel() + shift + 16, dtype=t.dtype, device="cuda")
    v = buf[shift:shift + t.numel()].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("shifts", [(0, 0, 0), (3, 3, 3), (0, 1, 2)])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,dim", [(5, 1), (4, 3), (9, 7), (3, 8), (7, 130), (5, 513), (2, 1025), (3, 4097), (2, 8200), (2, 16385),
                                      (2, 33001), (1, 70003), (1, 140001)])
def test_rows(rows, dim, dtype, shifts):
    print("softmax rows %dx%d %s shifts %s" % (rows, dim, dtype, shifts), flush=True)
    L, st = _capi.lib(), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device="cuda").manual_seed(rows * 31 + dim)
    x0, g0 = (torch.randn(rows, dim, device="cuda", generator=gen).to(TORCH_DTYPE[dtype]) for _ in range(2))
    xd = x0.double().cpu().numpy()
    m = xd.max(1, keepdims=True)
    e = np.exp(xd - m)
    soft, logs = e / e.sum(1, keepdims=True), xd - m - np.log(e.sum(1, keepdims=True))
    eps, fp = EPS[dtype], 2.0 ** -24
    for log, exp in ((0, soft), (1, logs)):
        x = placed(x0, shifts[0])
        for out in (placed(torch.zeros_like(x0), shifts[2]), x):  # apart, then over the input
            assert L.ttfused_softmax(CODE[dtype], x.data_ptr(), out.data_ptr(), rows, dim, 1, log, st) == 0
            torch.cuda.synchronize()
            # fp32 throughout: a few roundings of the exponent's argument and of the sum, then the type's own
            bound = eps * np.abs(exp) + fp * ((32 + np.abs(xd - m)) * soft if not log else 32 + np.abs(xd - m)) + (6e-8 if dtype == "f16" else 0)
            assert (np.abs(out.double().cpu().numpy() - exp) <= bound).all(), (log, out is x)
        y0 = torch.from_numpy(exp).cuda().to(TORCH_DTYPE[dtype])
        yd, gd = y0.double().cpu().numpy(), g0.double().cpu().numpy()
        dx = gd - np.exp(yd) * gd.sum(1, keepdims=True) if log else yd * (gd - (yd * gd).sum(1, keepdims=True))
        size = np.abs(gd).sum(1, keepdims=True) if log else (np.abs(yd * gd)).sum(1, keepdims=True)
        factor = np.exp(yd) if log else yd
        g, y = placed(g0, shifts[0]), placed(y0, shifts[1])
        for out in (placed(torch.zeros_like(x0), shifts[2]), g):
            assert L.ttfused_softmax_backward(CODE[dtype], g.data_ptr(), y.data_ptr(), out.data_ptr(), rows, dim, 1, log, st) == 0
            torch.cuda.synchronize()
            bound = eps * np.abs(dx) + fp * (8 * np.abs(gd) + (8 + np.abs(yd) + np.sqrt(dim) * 4) * np.abs(factor) * size) + (6e-8 if dtype == "f16" else 0)
            assert (np.abs(out.double().cpu().numpy() - dx) <= bound).all(), (log, "backward", out is g)
