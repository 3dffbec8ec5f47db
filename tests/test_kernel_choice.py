"""Which kernel a call runs on, as the host's queries answer without a GPU: sizes on either side of the rules that choose among kernels,
with what both sides measured on an MI355X."""
import ctypes

import pytest

from tinytorch_amd import _capi

F32, F16, BF16 = _capi.F32, _capi.F16, _capi.BF16
FAKE = 1 << 30  # an aligned address that nothing reads


def attention(dtype, B, Hq, Hkv, L, S, D, causal=False, mask=None, back=False):
    """Parameter block of dense tensors; mask: "keys" (Bool, one row for all), "bool" or "add" (a row each)."""
    bp = _capi.BackwardParams()
    _capi.lib().ttsdpa_backward_params_init(ctypes.byref(bp), dtype, B, Hq, Hkv, L, S, D)
    p = bp.fwd
    p.q = p.k = p.v = p.out = bp.dout = bp.dq = bp.dk = bp.dv = FAKE
    p.causal = _capi.CAUSAL_TOP_LEFT if causal else _capi.CAUSAL_NONE
    if mask:
        p.mask, p.mask_kind = FAKE, _capi.MASK_ADD if mask == "add" else _capi.MASK_BOOL
        for i, x in enumerate((S, 0, 0, 1) if mask == "keys" else (0, L * S, S, 1)):
            p.mask_stride[i] = x
    return bp if back else p


def test_queries_refuse_what_the_calls_refuse():
    L = _capi.lib()
    i, k = _capi.LinearKernelInfo(), ctypes.c_int(-1)
    assert L.ttlinear_matmul_kernel(7, 64, 64, 64, 0, 1, ctypes.byref(i)) == _capi.ERR_DTYPE
    assert L.ttlinear_matmul_kernel(BF16, 64, 0, 64, 0, 1, ctypes.byref(i)) == _capi.ERR_SHAPE
    assert L.ttlinear_matmul_kernel(BF16, 64, 64, 64, 0, 1, None) == _capi.ERR_NULL
    assert L.ttlinear_backward_kernels(BF16, 64, 64, 64, 1, ctypes.byref(i), None, ctypes.byref(k)) == _capi.ERR_NULL
    p = attention(BF16, 1, 3, 2, 64, 64, 64)
    assert L.ttsdpa_kernel(ctypes.byref(p), ctypes.byref(k)) == _capi.ERR_SHAPE
    bp = attention(BF16, 1, 2, 2, 64, 64, 64, back=True)
    bp.dout = None
    assert L.ttsdpa_backward_kernel(ctypes.byref(bp), 1 << 20, ctypes.byref(k)) == _capi.ERR_NULL


def test_ways_of_products():
    assert _capi.linear_kernel(BF16, 8192, 6144, 4096)[0] == "tiled"
    assert _capi.linear_kernel(BF16, 24, 2048, 5632) == ("stream", (16, 16), 1, 1)
    assert _capi.linear_kernel(BF16, 288, 2048, 6592) == ("tiled", (0, 0), 1, 5)     # divided
    assert _capi.linear_kernel(F16, 4096, 4096, 16, 1, 0)[0] == "outer"              # a weight's gradient of 16 rows
    assert _capi.linear_kernel(F32, 6, 768, 28672, 1, 1) == ("tiled", (0, 0), 1, 16)  # too narrow for the streaming kernel
    assert _capi.linear_kernel(F32, 3, 50, 70, 1, 0)[0] in ("general", "tiled")
    assert _capi.linear_backward_kernels(BF16, 8192, 4096, 4096)[2] is False
    assert _capi.linear_backward_kernels(F32, 64, 500, 784)[2] is True


# (the calls that the streaming kernel takes in fp32 add a contraction up in its chains)
@pytest.mark.parametrize("M,N,K", [(119, 3072, 9152), (300, 1021, 3200), (64, 512, 16384)])
def test_fp32_products_are_not_divided_into_longer_chains(M, N, K):
    assert _capi.linear_kernel(F32, M, N, K)[0] == "stream"


def test_kernels_of_short_sequences():
    assert _capi.kernel(attention(F32, 1, 4, 4, 128, 128, 64, causal=True)) == "short"
    assert _capi.backward_kernel(attention(F32, 1, 4, 4, 128, 128, 64, causal=True, back=True)) == "short_joint"
    assert _capi.kernel(attention(BF16, 2, 32, 8, 4096, 4096, 128, causal=True)) == "other"
    assert _capi.kernel(attention(F16, 16, 12, 12, 197, 197, 64, mask="keys")) == "heads_32"
    assert _capi.kernel(attention(F16, 1, 8, 8, 94, 94, 64, mask="keys")) == "heads_16"
    assert _capi.kernel(attention(F32, 1, 8, 8, 94, 94, 64, mask="keys")) == "other"
    bp = attention(BF16, 3, 4, 2, 100, 160, 64, causal=True, back=True)  # less scratch than asked for: the other kernels
    need = _capi.lib().ttsdpa_backward_workspace_bytes(ctypes.byref(bp))
    assert _capi.backward_kernel(bp) != "other" and _capi.backward_kernel(bp, need - 1) == "other"


@pytest.mark.parametrize("dtype,M,N,K,tile,tiles", [
    # backward of a layer, us, a tile of the weight's gradient to a workgroup / several
    (BF16, 24, 128, 192, 16, 1),     # 3.7 / 4.5: all tiles of both products run side by side
    (F16, 34, 128, 128, 16, 1),      # 3.7 / 4.5
    (BF16, 97, 320, 232, 32, 1),     # 4.2 / 5.0 (16 x 16): a round of larger ones
    (F32, 24, 512, 320, 32, 1),      # 5.4 / 7.7: fp32's share a CU in pairs
    (F32, 20, 40, 3328, 32, 1),      # 5.5 / 7.3
    (F32, 72, 576, 320, 32, 2),      # 6.7 / 6.0
    (F32, 64, 500, 784, 32, 4),      # more than a round
    (F32, 19, 2048, 2048, 32, 8),    # 55 / 21
])
def test_tiles_of_a_weights_gradient(dtype, M, N, K, tile, tiles):
    of_weight, _, one = _capi.linear_backward_kernels(dtype, M, N, K)
    assert one and of_weight == ("stream", (tile, tile), tiles, 1)


@pytest.mark.parametrize("M,N,K,way", [
    # us in one round of 64 x 64 tiles on the streaming kernel / divided among workgroups
    (539, 1600, 2432, "stream"),   # 14.1 / 18.1
    (444, 1920, 2624, "stream"),   # 14.4 / 18.0
    (865, 1024, 3328, "stream"),   # 17.6 / 19.4
    (288, 2048, 6592, "tiled"),    # 29.2 / 22.9
    (414, 2176, 9984, "tiled"),    # 49.0 / 36.8
])
def test_divided_where_one_round_of_small_tiles_is_longer(M, N, K, way):
    for dtype in (F16, BF16):
        kernel = _capi.linear_kernel(dtype, M, N, K)
        assert kernel[0] == way and (kernel[3] > 1) == (way == "tiled")


def test_whole_rounds_of_shares():
    for dtype in (F16, BF16):
        # us in one share and two: 32.7 and 35.2, 29.4 and 32.5
        assert _capi.linear_kernel(dtype, 54, 18688, 3072)[3] == 1
        assert _capi.linear_kernel(dtype, 276, 3864, 2800)[3] == 1
        # 44 tiles in four shares and eight, a round and a half: 16.8 and 21.1
        assert _capi.linear_kernel(dtype, 112, 1408, 8448)[3] == 4


@pytest.mark.parametrize("M,N,K,tile", [
    # us in 32 x 32 tiles / the smaller ones that were taken
    (1, 28672, 4096, (16, 16)),    # 45.1 / 42.5
    (8, 32000, 4096, (16, 16)),    # 55.3 / 48.7
    (6, 44032, 2560, (32, 32)),    # 0.91 of the speed in 16 x 16 ones
    (8, 50304, 3072, (32, 32)),    # 59.1 / 61.1
    (9, 28672, 4096, (32, 32)),
    (14, 15360, 5120, (32, 32)),   # 29.3 / 34.2
    (11, 16000, 3072, (32, 32)),   # 21.2 / 24.2
    (14, 10000, 3072, (32, 48)),   # of 16 x 16, 32 x 48 and 16 x 64 tiles the shortest, by 14 and 12 %
    (14, 10000, 4096, (16, 16)),
    (14, 10000, 2048, (16, 64)),
    (14, 16384, 2048, (16, 64)),
    (24, 8704, 4096, (32, 48)),
    (24, 12352, 4096, (32, 32)),
    (8, 8192, 4096, (32, 32)),
])
def test_tiles_of_few_rows(M, N, K, tile):
    for dtype in (F16, BF16):
        kernel = _capi.linear_kernel(dtype, M, N, K)
        assert kernel[0] == "stream" and kernel[1] == tile


@pytest.mark.parametrize("M,N,K,tile", [
    # us in 32 x 32 tiles / 16 x 32 ones, of a contraction-major weight
    (16, 8192, 2048, (16, 32)),   # 12.6 / 11.0
    (12, 7928, 2744, (32, 32)),   # 14.4 / 15.3: six units a wavefront
    (4, 4911, 3321, (16, 32)),    # 15.9 / 13.7
    (8, 5179, 3064, (32, 32)),    # 14.5 / 15.3
    (16, 5179, 3064, (32, 32)),   # 15.2 / 16.1
    (14, 6144, 4096, (16, 32)),
    (16, 8192, 1100, (32, 32)),
    (30, 11264, 4096, (32, 64)),
])
def test_tiles_of_few_rows_contraction_major(M, N, K, tile):
    for dtype in (F16, BF16):
        kernel = _capi.linear_kernel(dtype, M, N, K, 0, 0)
        assert kernel[0] == "stream" and kernel[1] == tile


@pytest.mark.parametrize("mask,B,H,L,D,kernel", [
    # us on the kernel for long sequences / on the one that holds a head's keys
    ("keys", 38, 16, 60, 32, "other"),     # 6.2 / 7.8: more than two rounds of workgroups
    ("keys", 43, 12, 22, 32, "other"),     # 5.4 / 6.7
    ("keys", 39, 16, 24, 16, "other"),     # 5.5 / 6.6
    ("keys", 39, 16, 23, 16, "heads_16"),  # 7.8 / 6.9: keys of no whole fours
    ("keys", 8, 12, 60, 32, "heads_16"),
    ("keys", 43, 12, 22, 64, "heads_16"),
    ("keys", 16, 12, 197, 64, "heads_32"),
    ("bool", 4, 8, 50, 32, "other"),       # 0.95 of the speed
    ("bool", 4, 8, 30, 48, "heads_16"),    # 1.2
    ("bool", 4, 8, 100, 32, "heads_16"),
    ("bool", 4, 8, 50, 64, "heads_16"),
    ("add", 8, 16, 128, 32, "other"),      # 6.5 / 7.7, its keys read four at a time
    ("add", 8, 16, 130, 32, "heads_16"),   # 8.5 / 6.2 at 93
    ("add", 46, 16, 20, 32, "heads_16"),   # 10.3 / 7.2
    ("add", 8, 16, 128, 64, "heads_16"),
])
def test_masked_heads(mask, B, H, L, D, kernel):
    for dtype in (F16, BF16):
        assert _capi.kernel(attention(dtype, B, H, H, L, L, D, mask=mask)) == kernel


@pytest.mark.parametrize("B,Hq,Hkv,L,D,kernel", [
    # fp32, causal: us on the kernel for long sequences / on the short sequences' one
    (1, 1, 1, 918, 128, "other"),   # 20.1 / 27.3
    (1, 1, 1, 892, 64, "other"),    # 14.5 / 15.8
    (2, 1, 1, 701, 64, "short"),    # 14.7 / 12.8
    (8, 32, 8, 76, 64, "other"),    # 12.1 / 14.6
    (4, 32, 4, 107, 128, "other"),  # 21.3 / 24.5
    (8, 4, 1, 435, 128, "other"),   # 33.5 / 38.6
    (4, 32, 8, 83, 64, "short"),    # 12.0 / 10.1
    (4, 32, 4, 75, 128, "short"),   # 19.4 / 17.9
    (1, 32, 8, 259, 128, "short"),  # 43.2 / 22.0
    (1, 16, 2, 652, 128, "short"),  # 50.4 / 38.4
    (8, 4, 4, 328, 128, "short"),   # 32.7 / 27.1: a head to every KV head
])
def test_fp32_forward_of_short_sequences(B, Hq, Hkv, L, D, kernel):
    assert _capi.kernel(attention(F32, B, Hq, Hkv, L, L, D, causal=True)) == kernel


@pytest.mark.parametrize("dtype,B,Hq,Hkv,L,D,kernel", [
    # causal, us on the kernels for long sequences / on the short sequences' one launch
    (F32, 4, 64, 8, 64, 64, "other"),          # 34.9 / 45.6
    (BF16, 4, 64, 8, 75, 64, "other"),         # 24.3 / 28.2
    (BF16, 8, 16, 2, 65, 128, "other"),        # 29.2 / 32.3
    (BF16, 2, 56, 8, 77, 128, "other"),        # 29.5 / 31.4
    (BF16, 8, 8, 8, 72, 64, "short_joint"),    # 15.0 / 14.4
    (BF16, 4, 16, 2, 124, 64, "short_joint"),  # 23.5 / 22.8
])
def test_backward_of_short_sequences_in_one_launch(dtype, B, Hq, Hkv, L, D, kernel):
    assert _capi.backward_kernel(attention(dtype, B, Hq, Hkv, L, L, D, causal=True, back=True)) == kernel
