"""Products over the experts' rows from a matrix of more rows than there are slots, whose last ones lie beyond 2 GiB."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [16, 64])             # (few rows an expert, and tiles)
def test_rows_beyond_two_gib(slots):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(slots)
    K, N, G = 2048, 128, 2
    T = (1 << 31) // (2 * K) + 64
    x = torch.zeros(T, K, dtype=torch.bfloat16, device="cuda")
    picked = torch.cat((torch.arange(T - slots // 2, T), torch.arange(slots - slots // 2)))
    x[picked.cuda()] = torch.randn(slots, K, generator=g).bfloat16().cuda()
    w = (torch.randn(G, N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    out = torch.empty(slots, N, dtype=torch.bfloat16, device="cuda")
    offsets = torch.tensor([0, slots // 2, slots], dtype=torch.int32, device="cuda")
    ops.experts_linear(x, picked.int().cuda(), w, offsets, out)
    rows = x[picked.cuda()].float()
    want = torch.cat((rows[: slots // 2] @ w[0].float().T, rows[slots // 2:] @ w[1].float().T))
    # (32-bit sums of 2048 products of order 2048 ** -0.5, then one rounding to bfloat16)
    assert bool(((out.float() - want).abs() <= 2.0 ** -8 * want.abs() + 2048 * 2.0 ** -24).all())
