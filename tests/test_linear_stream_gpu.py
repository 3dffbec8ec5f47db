"""The streaming product kernel (csrc/linear_stream.hip) at the edges of its tiles and units: every operand layout, rows
around the 16-row blocks, contractions around the 128-byte units and the eight wavefronts' turns, rows that begin at
any element, leading dimensions beyond the row; against the products of the same values in float64."""
import numpy as np
import pytest
import torch

from gpu_util import TORCH_DTYPE
from tinytorch_amd import _capi

pytestmark = pytest.mark.gpu

CODE = {"f32": _capi.F32, "f16": _capi.F16, "bf16": _capi.BF16}
# half a unit in the last place of the result's type, on top of K products summed in fp32 in any order
EPS = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def product(M, N, K, ta, tb, dtype, bias, pad=0, lead=0):
    """op(a) . op(b) + bias on operands `lead` elements into rows `pad` elements too long; -> nothing, asserts."""
    print("stream M%d N%d K%d tA%d tB%d %s bias%d pad%d lead%d" % (M, N, K, ta, tb, dtype, bias, pad, lead), flush=True)
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N * 3 + K)
    def operand(rows, cols):
        buf = torch.randn(rows, cols + pad + lead, device="cuda", generator=g).to(TORCH_DTYPE[dtype])
        return buf[:, lead:lead + cols]
    a, b = operand(*((K, M) if ta else (M, K))), operand(*((N, K) if tb else (K, N)))
    c = torch.randn(N, device="cuda", generator=g).to(TORCH_DTYPE[dtype]) if bias else None
    obuf = torch.full((M, N + 5), 7.0, device="cuda", dtype=TORCH_DTYPE[dtype])
    rc = _capi.lib().ttlinear_matmul(CODE[dtype], a.data_ptr(), b.data_ptr(), c.data_ptr() if bias else None, obuf.data_ptr(), M, N, K,
                                     int(ta), int(tb), a.stride(0), b.stride(0), N + 5, None, 0,
                                     torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0
    ad, bd = (t.double().cpu().numpy() for t in (a, b))
    ad, bd = ad.T if ta else ad, bd.T if tb else bd
    exp = ad @ bd + (c.double().cpu().numpy() if bias else 0)
    size = np.abs(ad) @ np.abs(bd) + (c.abs().double().cpu().numpy() if bias else 0)
    got = obuf[:, :N].double().cpu().numpy()
    assert (np.abs(got - exp) <= EPS[dtype] * np.abs(exp) + (K + 2) * 2.0 ** -24 * size + 1e-30).all(), np.abs(got - exp).max()
    assert (obuf[:, N:] == 7.0).all()  # nothing beyond the row


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("K", [1, 7, 31, 33, 63, 64, 65, 127, 509, 513, 777])
def test_contraction_edges(K, ta, tb, dtype):
    product(37, 29, K, ta, tb, dtype, bias=K % 2 == 1)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("M,N", [(1, 1), (1, 16), (16, 16), (17, 15), (31, 33), (64, 100), (65, 1001), (300, 70), (1001, 515)])
def test_row_edges(M, N, ta, tb, dtype):
    product(M, N, 130, ta, tb, dtype, bias=True)


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("pad,lead", [(1, 0), (3, 1), (8, 8)])
def test_leading_dimensions(pad, lead, ta, tb, dtype):
    product(50, 66, 200, ta, tb, dtype, bias=True, pad=pad, lead=lead)


@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False)])
def test_long_contraction(ta, tb):
    product(40, 48, 8192 + 3, ta, tb, "bf16", bias=False)


def test_batched_entries():
    """One launch for the entries of a batch, transposed operands of odd sizes."""
    from tinytorch_amd import matmul
    g = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randn(6, 5, 35, 51, device="cuda", generator=g)
    b = torch.randn(6, 5, 35, 43, device="cuda", generator=g)
    exp = a.double().cpu().numpy().swapaxes(-1, -2) @ b.double().cpu().numpy()
    got = matmul(a, b, True, False).double().cpu().numpy()
    assert np.abs(got - exp).max() <= 40 * 2.0 ** -24 * 35 * 4


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("M,K,N", [(1, 16, 16), (3, 17, 40), (64, 784, 500), (65, 130, 33), (200, 64, 1000), (1001, 515, 300),
                                   (7, 5, 9), (2100, 136, 72)])
def test_backward_of_a_layer(M, K, N, dtype):
    """Both gradients and the bias's: one launch for small layers (tiles of 16, 32 and 64), separate kernels for operands too
    narrow for it, column sums over several row ranges."""
    from tinytorch_amd import linearBackward
    print("layer backward M%d K%d N%d %s" % (M, K, N, dtype), flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    go, x, w = (torch.randn(*s, device="cuda", generator=g).to(TORCH_DTYPE[dtype]) for s in ((M, N), (M, K), (N, K)))
    got = linearBackward(go, x, w)
    god, xd, wd = (t.double().cpu().numpy() for t in (go, x, w))
    ones = np.ones((M, 1))
    for name, out, a, b in (("input", got[0], god, wd), ("weight", got[1], god.T, xd), ("bias", got[2][:, None], god.T, ones)):
        exp, size, n = a @ b, np.abs(a) @ np.abs(b), a.shape[1]
        err = np.abs(out.double().cpu().numpy() - exp)
        assert (err <= EPS[dtype] * np.abs(exp) + (n + 2) * 2.0 ** -24 * size + 1e-30).all(), (name, err.max())


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("M,N", [(1, 1), (63, 127), (65, 129), (1500, 200), (5000, 70), (8192, 1030)])
def test_column_sums(M, N, dtype):
    """The bias's gradient where it has a kernel of its own (a layer with 8 inputs is too narrow for the joint launch)."""
    from tinytorch_amd import linearBackward
    g = torch.Generator(device="cuda").manual_seed(M + N)
    go, x, w = (torch.randn(*s, device="cuda", generator=g).to(TORCH_DTYPE[dtype]) for s in ((M, N), (M, 8), (N, 8)))
    got = linearBackward(go, x, w)[2].double().cpu().numpy()
    god = go.double().cpu().numpy()
    exp, size = god.sum(0), np.abs(god).sum(0)
    assert (np.abs(got - exp) <= EPS[dtype] * np.abs(exp) + M * 2.0 ** -24 * size).all()
