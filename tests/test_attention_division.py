"""How attention calls are divided, as the host's queries answer without a GPU."""
import ctypes

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
