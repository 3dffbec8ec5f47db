"""How attention calls are divided, as the host's queries answer without a GPU."""
import ctypes
import time

import pytest

from tinytorch_amd import _capi

F32, F16, BF16 = _capi.F32, _capi.F16, _capi.BF16
FAKE = 1 << 30  # an aligned address that nothing reads
NONE, TL, BR = _capi.CAUSAL_NONE, _capi.CAUSAL_TOP_LEFT, _capi.CAUSAL_BOTTOM_RIGHT


def call(dtype, B, Hq, Hkv, L, S, D, causal=NONE, lens=False, back=False):
    bp = _capi.BackwardParams()
    _capi.lib().ttsdpa_backward_params_init(ctypes.byref(bp), dtype, B, Hq, Hkv, L, S, D)
    p = bp.fwd
    p.q = p.k = p.v = p.out = bp.dout = bp.dq = bp.dk = bp.dv = FAKE
    p.causal = causal
    if lens:
        p.kv_len = FAKE
    return bp if back else p


def scratch(p):
    L = _capi.lib()
    return (L.ttsdpa_backward_workspace_bytes if isinstance(p, _capi.BackwardParams) else L.ttsdpa_workspace_bytes)(ctypes.byref(p))


def test_queries_refuse_what_the_calls_refuse():
    L, n = _capi.lib(), ctypes.c_int(-1)
    assert L.ttsdpa_division(ctypes.byref(call(BF16, 1, 3, 2, 64, 64, 64)), ctypes.byref(n), None) == _capi.ERR_SHAPE
    bp = call(BF16, 1, 2, 2, 64, 64, 64, back=True)
    bp.dout = None
    assert L.ttsdpa_backward_division(ctypes.byref(bp), ctypes.byref(n), None) == _capi.ERR_NULL
    assert n.value == -1


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,D", [
    (1, 32, 8, 1, 1500, 128), (64, 32, 8, 1, 8192, 128), (24, 16, 8, 1, 1000, 64), (1, 4, 2, 700, 5000, 128), (1, 2, 2, 777, 777, 80),
    (2, 32, 8, 4096, 4096, 128), (1, 4, 4, 128, 128, 64), (1, 8, 8, 12, 3000, 128), (3, 4, 4, 5, 7, 20)])
def test_records_go_with_pieces(dtype, B, Hq, Hkv, L, S, D):
    """A call on the kernels for long sequences asks for scratch exactly where its keys are divided; in the backward beyond the rows'
    statistics."""
    p = call(dtype, B, Hq, Hkv, L, S, D)
    if _capi.kernel(p) in ("other", "dealt"):
        assert (_capi.division(p)[0] > 1) == (scratch(p) > 0)
    bp = call(dtype, B, Hq, Hkv, L, S, D, back=True)
    assert (max(_capi.backward_division(bp)) > 1) == (scratch(bp) > 16 * B * Hq * L)


@pytest.mark.parametrize("dtype,B,Hq,Hkv,S,D,lens,one,waves", [
    # us divided (or with four wavefronts) / in one launch (with eight), keys full, spread evenly and one long sequence among short ones
    (BF16, 32, 32, 8, 4096, 128, True, False, 4),    # 92.6 / 89.9, 64.2 / 70.7, 46.1 / 62.3
    (BF16, 32, 32, 8, 2048, 128, True, False, 4),    # 51.0 / 47.0, 35.7 / 37.2, 27.1 / 32.7
    (F32, 32, 32, 8, 1024, 128, True, False, 4),     # 47.9 / 44.5, 34.7 / 36.5, 26.1 / 31.5
    (BF16, 32, 32, 8, 1024, 128, True, True, 8),     # 29.4 / 24.8, 21.8 / 20.9, 17.1 / 17.6
    (F16, 24, 32, 8, 1024, 64, True, True, 8),       # 16.2 / 13.1, 13.9 / 11.6, 11.4 / 9.9
    (BF16, 32, 32, 8, 2048, 128, False, True, 8),    # 51.0 / 47.0
    (BF16, 64, 64, 8, 1024, 128, False, True, 4),    # 51.0 / 54.5
    (F16, 64, 64, 8, 4096, 64, False, True, 4),      # 93.2 / 94.3
    (F32, 69, 4, 4, 434, 128, True, None, 4),        # 32.9 / 35.4
    (BF16, 70, 16, 4, 1206, 80, True, False, 4),     # 35.8 / 41.7, 28.3 / 30.1, 16.5 / 19.3
    (F32, 21, 8, 2, 284, 80, True, False, 4),        # 13.7 / 16.3, 11.6 / 12.1, 10.5 / 13.3
])
def test_decode_in_one_launch(dtype, B, Hq, Hkv, S, D, lens, one, waves):
    """Where all keys of a sequence are one workgroup's, and of how many wavefronts: not where lengths may differ and the longest takes
    longer than its pieces and their merge."""
    pieces, w = _capi.division(call(dtype, B, Hq, Hkv, 1, S, D, lens=lens))
    assert w == waves
    assert one is None or (pieces == 1) == one


@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,causal,kernel,pieces", [
    # as summed up row tile by row tile
    (2, 2, 2, 2489, 2489, 64, NONE, "other", 5),
    (2, 2, 1, 6509, 6509, 128, NONE, "other", 2),
    (5, 2, 2, 357, 2647, 64, NONE, "dealt", 6),
    (1, 1, 1, 7821, 1760, 128, BR, "dealt", 4),
    (3, 6, 6, 871, 5902, 64, BR, "dealt", 2),
    (1, 10, 5, 7210, 7054, 128, TL, "dealt", 1),
    (1, 3, 3, 1569, 1300, 128, TL, "dealt", 6),
    (7, 1, 1, 3440, 3440, 64, BR, "other", 4),
    (3, 3, 3, 4128, 4128, 64, BR, "dealt", 1),
    (1, 9, 9, 231, 868, 64, BR, "other", 5),
    (2, 4, 1, 8721, 8721, 64, BR, "dealt", 1),
    (6, 2, 2, 2418, 2418, 128, TL, "dealt", 1),
    (1, 22, 11, 806, 2578, 64, BR, "dealt", 1),
    (4, 2, 2, 1231, 6702, 64, BR, "other", 6),
    (1, 16, 16, 1112, 1112, 64, TL, "dealt", 1),
    (7, 2, 1, 2722, 2722, 64, TL, "dealt", 1),
    (1, 16, 4, 383, 866, 64, BR, "other", 3),
    (2, 4, 1, 8980, 8980, 128, TL, "dealt", 1),
    (1, 6, 3, 2290, 2290, 128, BR, "dealt", 3),
    (1, 1, 1, 785, 2221, 128, BR, "dealt", 9),
    (3, 2, 1, 1553, 1553, 128, BR, "dealt", 4),
    (4, 1, 1, 1439, 1439, 64, NONE, "dealt", 3),
    (2, 24, 6, 1341, 6526, 64, NONE, "dealt", 1),
    (1, 1, 1, 1182, 1182, 128, TL, "dealt", 5),
])
def test_pieces_of_a_prompt(B, Hq, Hkv, L, S, D, causal, kernel, pieces):
    """The row tiles' lengths in closed form: rows and keys that end anywhere, both alignments, more rows than keys."""
    p = call(BF16, B, Hq, Hkv, L, S, D, causal)
    assert (_capi.kernel(p), _capi.division(p)[0]) == (kernel, pieces)


def test_planning_does_not_grow_with_the_rows():
    """Host time of a scratch query for 16 to 64 times the rows (row tile by row tile 9 and 2 times as long)."""
    def least(f, p):
        ref, times = ctypes.byref(p), []
        for _ in range(60):
            t = time.perf_counter()
            for _ in range(100):
                f(ref)
            times.append(time.perf_counter() - t)
        return min(times)
    L = _capi.lib()
    f, g = L.ttsdpa_workspace_bytes, L.ttsdpa_backward_workspace_bytes
    assert least(f, call(BF16, 1, 1, 1, 16384, 16384, 128, TL)) < 3 * least(f, call(BF16, 1, 1, 1, 1100, 1100, 128, TL))
    assert least(g, call(BF16, 1, 1, 1, 65536, 65536, 128, TL, back=True)) < 1.5 * least(g, call(BF16, 1, 1, 1, 1100, 1100, 128, TL, back=True))


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,D", [
    # us with the row blocks' keys counted as if all were seen / counted as they are
    (1, 4, 4, 130, 817, 64),       # 26.3 / 18.5
    (2, 4, 2, 187, 1230, 64),      # 33.0 / 24.5
    (1, 8, 4, 1776, 6154, 64),     # 78.2 / 78.2
    (2, 8, 4, 174, 1758, 128),     # 38.3 / 29.7
    (1, 32, 8, 300, 4000, 128),    # 73 / 62
    (4, 1, 1, 1401, 17781, 128),   # 75.1 / 68.5
])
def test_row_blocks_of_a_top_left_mask_see_as_many_keys_as_rows(dtype, B, Hq, Hkv, L, S, D):
    assert _capi.backward_division(call(dtype, B, Hq, Hkv, L, S, D, TL, back=True))[1] == _capi.backward_division(call(dtype, B, Hq, Hkv, L, L, D, TL, back=True))[1]


@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,causal,pieces", [
    (1, 16, 2, 1031, 1031, 64, BR, (14, 3)),       # us with dk / dv in 8 pieces 71.3, in 14 58.5
    (1, 32, 8, 4528, 111, 128, BR, (15, 1)),       # 128.9, 105.4
    (2, 2, 1, 421, 6630, 128, NONE, (1, 14)),      # dq in 8 75.3, in 14 71.1
    (1, 8, 8, 263, 4859, 64, BR, (1, 8)),          # in 14 52.4, in 8 49.4
    (4, 2, 1, 424, 3598, 64, BR, (2, 8)),          # in 10 57.5, in 8 54.4
    (4, 64, 8, 211, 1711, 64, TL, (3, 1)),         # dk / dv whole 85, in three pieces, of whose records most are zeros, 67
    (2, 64, 8, 841, 7870, 128, TL, (1, 1)),        # 217, in two pieces 248: more than the caches hold
])
def test_pieces_of_long_streams(B, Hq, Hkv, L, S, D, causal, pieces):
    for dtype in (F16, BF16):
        assert _capi.backward_division(call(dtype, B, Hq, Hkv, L, S, D, causal, back=True)) == pieces


# ---- what the GPU tests' cases are meant for: held here, where the estimates are ---------------------------------------------------------------
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,causal,lens,divided", [
    (1, 4, 2, 700, 5000, BR, False, True), (1, 4, 2, 1100, 3000, BR, False, True),
    (3, 4, 2, 700, 3000, BR, True, True),                                             # (there in pages)
    (1, 16, 4, 650, 650, TL, False, False), (4, 8, 8, 514, 545, NONE, True, False)])  # weightless rows; key counts
def test_dealt_cases(B, Hq, Hkv, L, S, causal, lens, divided, dtype, D):
    """test_prefill_dealt_gpu.py: the rows said to be divided are, and the test of infinities beyond the diagonal runs on that kernel."""
    p = call(dtype, B, Hq, Hkv, L, S, D, causal, lens)
    assert _capi.kernel(p) == "dealt" and (_capi.division(p)[0] > 1) == divided


def test_backward_cases():
    """test_backward_streams_gpu.py: divided key ranges; query streams in a number of pieces that is no power of two, over more workgroups than
    run side by side; whole ones too."""
    def pieces(*a, D=128, causal=NONE):
        bp = call(BF16, *a, D, causal, back=True)
        assert _capi.backward_kernel(bp) == "other"
        return _capi.backward_division(bp)
    assert pieces(2, 2, 1, 129, 2111)[1] > 1 and pieces(1, 8, 4, 200, 1500, causal=BR)[1] > 1
    few = [pieces(1, Hq, Hkv, L, 1230, causal=c) for Hq, Hkv in ((6, 2), (5, 5), (7, 1)) for L in (33, 64, 96, 160, 193) for c in (NONE, BR)]
    assert any(n > 1 and m > 1 for n, m in few) and any(n == 1 and m > 1 for n, m in few)
    walks = [pieces(*a, D=D, causal=TL)[0] for D in (128, 64) for a in ((4, 56, 8, 383, 383), (4, 32, 4, 909, 909), (2, 32, 8, 700, 700))]
    assert all(n > 1 for n in walks) and any(n & (n - 1) for n in walks)


def test_decode_cases():
    """test_decode_one_launch_gpu.py: workgroups of eight wavefronts for every type and head size there, and calls that stay divided."""
    for D, dtype in ((128, BF16), (64, F16), (80, BF16), (128, F32), (64, F32)):
        assert _capi.division(call(dtype, 2, 10, 2, 1, 256, D)) == (1, 8)
    assert _capi.division(call(F32, 2, 6, 2, 1, 257, 128)) == (3, 4) and _capi.division(call(BF16, 2, 16, 2, 1, 289, 128)) == (3, 4)
    for D, dtype in ((128, BF16), (64, F16), (64, F32)):
        assert _capi.division(call(dtype, 24, 16, 8, 1, 1000, D, lens=True)) == (1, 8)
