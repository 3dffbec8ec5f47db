"""The order in which a decode wavefront adds its value lanes' sums: the keys of a load instruction (64 lanes / chunks of a row) in pairs of
neighbours, then pairs of pairs.  All scores are zero, so every probability is one; large values cancel only if they meet in that order, and
the small one left over is exact."""
import pytest
import torch

from gpu_util import TORCH_DTYPE, call

pytestmark = pytest.mark.gpu

S = 256
# 24 bits and more between the two: a sum of both keeps the large one alone
LARGE = {"bf16": (2.0 ** 30, 1.0), "f16": (2.0 ** 15, 2.0 ** -10), "f32": (2.0 ** 30, 1.0)}


@pytest.mark.parametrize("D,dtype,phases", [(128, "bf16", 4), (128, "f16", 4), (80, "bf16", 4), (64, "bf16", 8), (64, "f16", 8), (40, "f16", 8), (64, "f32", 4)])
@pytest.mark.parametrize("G", [1, 5])
@pytest.mark.parametrize("apart", [1, 2, 4])
def test_neighbours_first(D, dtype, phases, G, apart):
    """The large ones `apart` keys from each other, the small one among the keys that are added after they have met."""
    if 2 * apart > phases:
        pytest.skip("more keys than a load instruction has")
    large, small = LARGE[dtype]
    q = torch.zeros(1, G, 1, D, dtype=TORCH_DTYPE[dtype], device="cuda")
    k = torch.randn(1, 1, S, D, device="cuda").to(q.dtype)
    v = torch.zeros_like(k)
    v[:, :, 0], v[:, :, apart] = large, -large
    if 2 * apart < phases:
        v[:, :, 2 * apart] = small
        expect = small / S
    else:  # the last addition of all: each side's small one is lost beside its large one
        v[:, :, 1] = small
        expect = 0.0
    rc, out = call("decode" if dtype != "f32" else "forward", q, k, v)
    assert rc == 0
    assert (out == expect).all(), out.float().unique()
