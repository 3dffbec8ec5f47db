"""attnMasks whose rows do not begin at groups of four keys, on the matrix-core kernels: key counts around the edges of a
mask block (groups of 4, blocks of 32, tiles of 64), strided keys, and per-batch key counts beside a mask."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import TOL, call, make_inputs, to_device, to_host_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["bool", "add"])
@pytest.mark.parametrize("dtype,D", [("f16", 64), ("bf16", 80), ("bf16", 128), ("f32", 64)])
@pytest.mark.parametrize("S", [1, 3, 5, 31, 33, 62, 65, 129, 203])
def test_odd_key_counts(S, dtype, D, kind):
    B, Hq, Hkv, L = 2, 4, 2, 37
    print("odd mask S%d %s D%d %s" % (S, dtype, D, kind), flush=True)
    host, dev = make_inputs(8800 + S, B, Hq, Hkv, L, S, D, dtype)
    rng = np.random.default_rng(S)
    if kind == "bool":
        m = rng.random((B, 1, L, S)) > 0.4
        m[..., S // 2] = True
        mh, md = m.astype(np.uint8), torch.from_numpy(m).cuda()
    else:
        mh, bits = oracle.round_to(rng.standard_normal((Hq, L, S)).astype(np.float32), dtype)
        md = to_device(mh, bits, dtype)
    rc, out = call("forward", *dev, mask=md)
    assert rc == 0
    assert np.abs(to_host_f32(out) - oracle.sdpa_f32(*host, mask=mh)).max() <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_strided_mask_and_key_counts(dtype):
    B, Hq, Hkv, L, S, D = 3, 4, 4, 70, 77, 64
    print("strided mask, key counts %s" % dtype, flush=True)
    host, dev = make_inputs(8900, B, Hq, Hkv, L, S, D, dtype)
    m = np.random.default_rng(5).random((S, L)) > 0.3
    m[0] = True
    md = torch.from_numpy(m).cuda().t()  # keys strided by L
    lens = [77, 34, 1]
    kv = torch.tensor(lens, dtype=torch.int32, device="cuda")
    rc, out = call("forward", *dev, mask=md, kv_lens=kv)
    assert rc == 0
    for b, n in enumerate(lens):
        exp = oracle.sdpa_f32(host[0][b:b + 1], host[1][b:b + 1, :, :n], host[2][b:b + 1, :, :n],
                              mask=np.ascontiguousarray(m.T[:, :n]).astype(np.uint8))
        assert np.abs(to_host_f32(out[b:b + 1]) - exp).max() <= TOL[dtype], b
