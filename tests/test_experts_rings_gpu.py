"""Products over the experts' rows through rings in shared memory: 32 weight rows and 16 slots a work-group at the edges of its tiles (slots 0, 1, 8, 9, 16, 17 and 33 of a group, columns that
end inside a block, one slab of K and more than a ring holds), and the dispatch around its lines on the slots a group has on average."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [0, 6])
@pytest.mark.parametrize("counts,N,K,act", [([0, 1, 8, 9, 16, 17, 33], 70, 64, "none"), ([17, 0, 15], 130, 1344, "silu_pairs"), ([5], 31, 2048, "relu2"), ([1] * 70, 32, 192, "gelu")])
def test_rings_over_groups_of_rows(which, counts, N, K, act):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(N + K)
    S, tokens = sum(counts), 23
    offsets = torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32).cuda()
    w = (torch.randn(len(counts), N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    x = torch.randn(tokens, K, generator=g).bfloat16().cuda()
    src = torch.randint(0, tokens, (S + 2,), generator=g, dtype=torch.int32).cuda()
    cols = N // 2 if act.endswith("_pairs") else N
    out = torch.full((S + 2, cols), 7.0, dtype=torch.bfloat16, device="cuda")
    want = torch.full_like(out, 7.0)
    ops.experts_linear_variant(x, src, w, offsets, out, act, which)
    ops.experts_linear(x, src, w, offsets, want, act, general=True)
    assert bool((out[S:] == 7.0).all())
    # both round sums of the same products once: at most neighbouring bfloat16 numbers, and near zero the sums' own error
    torch.testing.assert_close(out.float(), want.float(), rtol=2.0 ** -7, atol=4 * K * 2.0 ** -24)


@pytest.mark.parametrize("K", [1984, 2048])
@pytest.mark.parametrize("slots", [1, 12, 13, 24, 25, 36, 37])
def test_the_dispatch_around_the_rings(K, slots):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(slots)
    G, N = 3, 48
    x, w = torch.randn(slots, K, generator=g).bfloat16().cuda(), (torch.randn(G, N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    counts = torch.bincount(torch.randint(0, G, (slots,), generator=g), minlength=G)
    offsets = torch.cat((torch.zeros(1, dtype=torch.long), counts.cumsum(0))).int().cuda()
    got, want = torch.empty(slots, N, dtype=torch.bfloat16, device="cuda"), torch.empty(slots, N, dtype=torch.bfloat16, device="cuda")
    ops.experts_linear(x, None, w, offsets, got)
    ops.experts_linear(x, None, w, offsets, want, general=True)
    torch.testing.assert_close(got.float(), want.float(), rtol=2.0 ** -7, atol=4 * K * 2.0 ** -24)


def test_more_groups_than_a_launch_has_tiles_of_eight_slots():
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(2)
    G, N, K, slots = 52000, 8, 2048, 4 * 52000
    w = torch.randn(G, N, K, device="cuda", dtype=torch.bfloat16) / K ** 0.5
    x, src = torch.randn(64, K, generator=g).bfloat16().cuda(), torch.randint(0, 64, (slots,), generator=g, dtype=torch.int32).cuda()
    offsets = (4 * torch.arange(G + 1)).int().cuda()
    got = torch.empty(slots, N, dtype=torch.bfloat16, device="cuda")
    ops.experts_linear(x, src, w, offsets, got)
    for e in (0, 1, 43700, 51999):
        want = x[src[4 * e: 4 * e + 4].long()].double() @ w[e].double().T
        torch.testing.assert_close(got[4 * e: 4 * e + 4].double(), want, rtol=2.0 ** -8, atol=1e-4)
