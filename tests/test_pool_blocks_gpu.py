"""Pooled blocks whose positions are fetched sixteen at a time: the sums of the positions one after the other, to the bit."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


# fewer than one group of positions, one, one and a rest, several; blocks that cross pages and that begin inside one; a position without a page
@pytest.mark.parametrize("pool", [1, 6, 15, 16, 17, 64])
@pytest.mark.parametrize("page", [8, 16])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hole", [False, True])
def test_means_in_the_order_of_the_positions(pool, page, dtype, hole):
    g = torch.Generator().manual_seed(pool + page)
    G, dim, vdim, ctx, n = 2, 36, 20, pool // 2, 3 * pool + 2
    pages = -(-(ctx + n) // page) + 3
    k = torch.randn(pages, G, page, dim, generator=g).to(dtype)
    v = torch.randn(pages, G, vdim, page, generator=g).to(dtype)
    table = (torch.randperm(pages - 1, generator=g)[: -(-(ctx + n) // page)] + 1).to(torch.int32)[None]
    if hole:
        table[0, 0] = 0
    pool_table = torch.tensor([[2, 1]], dtype=torch.int32)
    pk, pv = torch.full((3, G, page, dim), 7.0, dtype=dtype), torch.full((3, G, vdim, page), 7.0, dtype=dtype)
    got_k, got_v = pk.cuda(), pv.cuda()
    ops.pool_blocks(k.cuda(), v.cuda(), table.cuda(), got_k, got_v, pool_table.cuda(), torch.tensor([0, n], dtype=torch.int32).cuda(),
                    torch.tensor([ctx], dtype=torch.int32).cuda(), n // pool + 1, page, pool)
    for b in range(ctx // pool, (ctx + n) // pool):
        ks, vs = torch.zeros(G, dim), torch.zeros(G, vdim)
        for p in range(b * pool, (b + 1) * pool):
            at = int(table[0, p // page])
            if at:
                ks, vs = ks + k[at, :, p % page].float(), vs + v[at, :, :, p % page].float()
        pk[int(pool_table[0, b // page]), :, b % page] = (ks / pool).to(dtype)
        pv[int(pool_table[0, b // page]), :, :, b % page] = (vs / pool).to(dtype)
    assert torch.equal(got_k.cpu(), pk) and torch.equal(got_v.cpu(), pv)
