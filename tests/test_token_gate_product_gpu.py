"""The product whose columns are gated with the token's own numbers (one launch up to 16 rows) against the product and the gate one after the other: the same bits; ids that are no
row of the table leave their outputs as they are."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17])
@pytest.mark.parametrize("N,K", [(256, 2048), (13, 64), (130, 448), (5000, 128), (40, 72)])
@pytest.mark.parametrize("activation", ["gelu_tanh", "silu"])
def test_product_gated_with_the_tokens_numbers(rows, N, K, activation):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(rows + N)
    x = torch.randn(rows, K + 8, generator=g).bfloat16().cuda()[:, :K]
    w = (torch.randn(N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    table = torch.randn(50, 3 * N, generator=g).bfloat16().cuda()[:, N: 2 * N]
    ids = torch.randint(0, 50, (rows,), generator=g).int()
    if rows > 2:
        ids[1], ids[2] = -1, 50
    z = torch.empty(rows, N, dtype=torch.float32, device="cuda")
    want, got = (torch.full((rows, N), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ops.linear(x, w, None, z)
    ops.token_gate(z, ids.cuda(), table, want, activation)
    ops.linear_token_gate(x, w, ids.cuda(), table, got, activation)
    assert torch.equal(got, want)
    if rows > 2:
        assert bool((got[1:3] == 7.0).all())
    with pytest.raises(ops.KernelError):
        ops.linear_token_gate(x, w, ids.cuda(), table[:, 1:], got, activation)
