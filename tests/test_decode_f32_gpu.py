"""fp32 on the split-KV streaming kernel: few query rows per KV head against a cache, with the scratch that lets the keys be
divided; head sizes at and between the kernel's, row counts up to its sixteen, strided queries, per-batch key counts, pages."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import TOL, call, make_inputs, max_abs_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,L,S,D", [(1, 1, 1, 1, 1, 64), (2, 4, 4, 1, 33, 128), (2, 8, 2, 1, 700, 128), (1, 8, 1, 2, 1500, 64),
                                            (3, 12, 4, 3, 513, 128), (2, 6, 2, 1, 300, 40), (2, 4, 1, 4, 900, 100)])
def test_few_rows(B, Hq, Hkv, L, S, D):
    print("f32 decode B%d %d/%d L%d S%d D%d" % (B, Hq, Hkv, L, S, D), flush=True)
    host, dev = make_inputs(9100 + S, B, Hq, Hkv, L, S, D, "f32")
    rc, out = call("forward", *dev)
    assert rc == 0
    assert max_abs_err(out, oracle.sdpa_f32(*host)) <= TOL["f32"]


@pytest.mark.parametrize("page", [0, 64])
def test_strided_queries_and_key_counts(page):
    B, Hq, Hkv, S, D = 4, 8, 2, 640, 128
    print("f32 decode, strided q, key counts, page %d" % page, flush=True)
    host, dev = make_inputs(9200, B, Hq, Hkv, 1, S, D, "f32")
    qkv = torch.randn(B, 1, Hq + 4, D, device="cuda")
    qkv[:, :, :Hq] = dev[0].transpose(1, 2)
    q = qkv.transpose(1, 2)[:, :Hq]
    lens = [640, 1, 65, 0]
    kv = torch.tensor(lens, dtype=torch.int32, device="cuda")
    k, v, table = dev[1], dev[2], None
    if page:
        n = S // page
        table = torch.randperm(B * n, device="cuda").to(torch.int32).view(B, n)
        pool = lambda t: torch.empty(B * n, Hkv, page, D, device="cuda").index_copy_(
            0, table.view(-1).long(), t.view(B, Hkv, n, page, D).transpose(1, 2).reshape(B * n, Hkv, page, D))
        k, v = pool(k), pool(v)
    rc, out = call("forward", q, k, v, kv_lens=kv, block_table=table)
    assert rc == 0
    for b, n in enumerate(lens):
        if n == 0:
            assert torch.count_nonzero(out[b]) == 0
            continue
        exp = oracle.sdpa_f32(host[0][b:b + 1], host[1][b:b + 1, :, :n], host[2][b:b + 1, :, :n])
        assert max_abs_err(out[b:b + 1], exp) <= TOL["f32"], b
