"""The Python entry points' two ways to the C ABI, the native binding and the Python code behind it: the same results for every
call that the native one takes, and other threads at work while it allocates and launches."""
import sys
import threading
import time

import pytest
import torch

import tinytorch_amd as tt
from tinytorch_amd import _native, function

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


class Nothing:
    """A binding that takes no call."""

    def __getattr__(self, name):
        assert hasattr(_native, name)
        return lambda *args: None


def calls(dtype):
    """(name, what the native binding has to take, a call of fresh arguments -> tensors)"""
    g = torch.Generator(device="cuda").manual_seed(11)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(DT[dtype])
    q, k, v = r(2, 8, 70, 64), r(2, 2, 130, 64), r(2, 2, 130, 64)
    lens = torch.tensor([130, 50], dtype=torch.int32, device="cuda")
    mask = torch.rand(70, 130, generator=g, device="cuda") < 0.7
    mask[:, 0] = True
    bias = r(8, 70, 130)
    go = r(2, 8, 70, 64)
    step = r(2, 1, 8, 64).transpose(1, 2)
    pool_k, pool_v = r(6, 2, 64, 64), r(6, 2, 64, 64)
    table = torch.tensor([[5, 0, 2], [1, 4, 3]], dtype=torch.int32, device="cuda")
    paged = torch.tensor([150, 64], dtype=torch.int32, device="cuda")
    x, w, b = r(33, 100), r(77, 100), r(77)
    gain, grad = r(100), r(33, 77)
    att = lambda *a, **kw: (lambda: tt.sdpAttention(*a, **kw))
    out = tt.sdpAttention(q, k, v, isCausal=True)
    out_m = tt.sdpAttention(q, k, v, attnMask=bias, scale=0.2)

    def append(table_arg, positions):
        kc, vc = (pool_k.clone(), pool_v.clone()) if table_arg is not None else (k.clone(), v.clone())
        new_k, new_v = q[:, :2, :3], q[:, 2:4, :3]
        tt.kvCacheAppend(kc, vc, new_k, new_v, positions, table_arg)
        return kc, vc

    def add_norm():
        a, res = x.clone(), x.flip(0).contiguous()
        tt.fusedAddRmsNorm(a, res, gain, 1e-5)
        return a, res

    return [
        ("sdp_attention", att(q, k, v)), ("sdp_attention", att(q, k, v, isCausal=True, causalAlign="bottom-right", kvLens=lens)),
        ("sdp_attention", att(q, k, v, attnMask=mask)), ("sdp_attention", att(q, k, v, attnMask=bias, scale=0.2)),
        ("sdp_attention", att(step, k, v, kvLens=lens)), ("sdp_attention", att(step, pool_k, pool_v, kvLens=paged, blockTable=table)),
        ("sdp_attention_backward", lambda: tt.sdpAttentionBackward(go, q, k, v, out, isCausal=True)),
        ("sdp_attention_backward", lambda: tt.sdpAttentionBackward(go, q, k, v, out_m, attnMask=bias, scale=0.2)),
        ("kv_cache_append", lambda: append(None, 5)), ("kv_cache_append", lambda: append(None, lens - 20)),
        ("kv_cache_append", lambda: append(table, paged - 3)),
        ("rms_norm", lambda: tt.rmsNorm(x, [100], gain, 1e-5)), ("rms_norm", lambda: tt.rmsNorm(x, (100,))), ("fused_add_rms_norm", add_norm),
        ("silu_mul", lambda: tt.siluMul(x)), ("softmax", lambda: tt.softmax(x, 0)), ("softmax", lambda: tt.logSoftmax(q, -1)),
        ("softmax_backward", lambda: tt.softmaxBackward(x, tt.softmax(x))), ("softmax_backward", lambda: tt.logSoftmaxBackward(x, tt.logSoftmax(x, -1), -1)),
        ("linear", lambda: tt.linear(x, w, b)), ("linear", lambda: tt.linear(x.view(3, 11, 100), w)),
        ("matmul", lambda: tt.matmul(x, w, False, True, b)), ("matmul", lambda: tt.matmul(x, x, True, False)),
        ("linear_backward", lambda: tt.linearBackward(grad, x, w)), ("linear_backward", lambda: tt.linearBackward(grad, x, w, needBias=False)),
    ]


# Both ways make the same launches, except: linearBackward, whose Python way is two products and torch's column sums, linear, whose
# Python way has no scratch to divide a contraction with (other orders of fp32 sums of up to 100 products, then one rounding)
SAME = {"linear": {"f32": 1e-6, "f16": 2e-3, "bf16": 1.6e-2}, "linear_backward": {"f32": 1e-6, "f16": 2e-3, "bf16": 1.6e-2}}


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_both_ways_agree(dtype, monkeypatch):
    for name, call in calls(dtype):
        print(name, flush=True)
        taken = []
        monkeypatch.setattr(function, "_native", type("Seen", (), {"__getattr__": lambda self, n: lambda *a: taken.append((n, getattr(_native, n)(*a))) or taken[-1][1]})())
        native = call()
        assert any(n == name and r is not None for n, r in taken), "the native binding left a call in order to Python: " + name
        monkeypatch.setattr(function, "_native", Nothing())
        python = call()
        monkeypatch.undo()
        native, python = ([t for t in (o if isinstance(o, tuple) else (o,)) if t is not None] for o in (native, python))
        assert len(native) == len(python)
        for a, b in zip(native, python):
            assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
            if name in SAME:
                assert ((a - b).norm() / b.norm()).item() <= SAME[name][dtype], name
            else:
                assert torch.equal(a, b), name


@pytest.mark.parametrize("what", ["rmsNorm", "linear", "sdpAttention"])
def test_other_threads_run_meanwhile(what):
    """With the interpreter's own switching out of the way, another thread gets its turns while the binding is at work."""
    x, w, q = torch.randn(4, 256, device="cuda"), torch.randn(8, 256, device="cuda"), torch.randn(1, 2, 16, 64, device="cuda")
    call = {"rmsNorm": lambda: _native.rms_norm(x, [256], None, 1e-5), "linear": lambda: _native.linear(x, w, None),
            "sdpAttention": lambda: _native.sdp_attention(q, q, q, False, None, 0.0, None, None, "top-left", None)}[what]
    assert call() is not None
    torch.cuda.synchronize()
    turns, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)  # gives the interpreter back

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other, daemon=True)
    thread.start()
    try:
        sys.setswitchinterval(1000)
        before = turns[0]
        for _ in range(3000):
            call()
        during = turns[0] - before
    finally:
        sys.setswitchinterval(interval)
        stop.set()
    thread.join()
    torch.cuda.synchronize()
    assert during >= 3000, during  # a turn for each call (some 45000; where the binding keeps the interpreter, 0 to 200 from before the loop)
