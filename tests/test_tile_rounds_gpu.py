"""Products of more than 128 rows whose tiles are one round of work-groups, and products that give one float slab."""
import math

import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    return x, w, x.double() @ w.double().T


# 256 tiles of 128 x 128 exactly, one row and one column less and more, one slab of K and a few
@pytest.mark.parametrize("M,N", [(2048, 2048), (2047, 2047), (2049, 2049), (1024, 4096), (129, 200), (750, 4104)])
@pytest.mark.parametrize("K", [64, 128, 320, 2048])
@pytest.mark.parametrize("result", [torch.bfloat16, torch.float32])
def test_one_round_of_tiles(M, N, K, result):
    x, w, ref = _operands(M, N, K)
    out = torch.full((M, N + 8), 7.0, dtype=result, device="cuda")
    ops.linear(x, w, None, out[:, :N])
    # (sums of K products in 32 bits, then one rounding of the result)
    atol = 8 * 2 ** -24 * math.sqrt(K)
    torch.testing.assert_close(out[:, :N].double(), ref, rtol=2 ** -8 if result == torch.bfloat16 else 2e-5, atol=atol)
    assert (out[:, N:] == 7.0).all()


# one slab (of 64 x 64 and of 128 x 128 tiles) and several: the slabs' sum is the product, and 32 bits are kept
@pytest.mark.parametrize("M,N,K,slabs", [(200, 3584, 3584, 1), (400, 7168, 3584, 1), (1457, 2048, 5632, 2), (400, 7168, 5120, 2), (1457, 2048, 4096, 2), (513, 5120, 5120, 2), (512, 5120, 13824, 3),
                                         (100, 4608, 3584, 7)])
def test_float_slabs(M, N, K, slabs):
    assert ops.linear_partials_pay(M, N, K)
    x, w, ref = _operands(M, N, K)
    got = ops.linear_partials(x, w)
    assert got.dtype == torch.float32 and got.shape == (slabs, M, N)
    torch.testing.assert_close(got.double().sum(0), ref, rtol=2e-5, atol=8 * 2 ** -24 * math.sqrt(K))
