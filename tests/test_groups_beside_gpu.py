"""Products of equal shape and one more beside them in one launch (up to 16 rows): the first with the bits that they have alone, the other one against 64 bits; the sizes that it is not
built for go one after the other."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17])
@pytest.mark.parametrize("groups,N,n,K", [(4, 2048, 64, 2048), (2, 100, 13, 64), (1, 40, 40, 192), (3, 24, 30, 128), (2, 64, 8, 72), (4, 1024, 160, 448)])
def test_products_and_one_more_beside_them(rows, groups, N, n, K):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(rows + N + K)
    mixes = torch.randn(groups + 1, rows, K, generator=g).bfloat16().cuda()
    w, w2 = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((groups, N, K), (n, K)))
    wide, want = (torch.full((rows, groups * N + 8), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    z = torch.full((rows + 1, n), 7.0, dtype=torch.float32, device="cuda")
    ops.linear_groups(mixes[:groups], w, want[:, : groups * N])
    ops.linear_groups_beside(mixes[:groups], w, wide[:, : groups * N], mixes[groups], w2, z[:rows])
    assert torch.equal(wide, want) and bool((z[rows] == 7.0).all())
    x, m = mixes[groups].double().cpu(), w2.double().cpu()
    bound = K * 2.0 ** -24 * (x.abs() @ m.abs().T)                  # (products of bfloat16 are exact in 32 bits; K additions)
    assert bool(((z[:rows].double().cpu() - x @ m.T).abs() <= bound).all())
    with pytest.raises(ops.KernelError):
        ops.linear_groups_beside(mixes[:groups], w, wide[:, : groups * N], mixes[groups], w2, z[:rows, : n - 1])
