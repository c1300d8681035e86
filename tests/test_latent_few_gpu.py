"""The latents' norms, rotation and cache write on both sides of 512 tokens (below: a work-group for each of them), against plain 64-bit formulas."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 511, 512])
@pytest.mark.parametrize("q_rank,rank,rot,dims,heads,halves", [(2056, 72, 24, 16, 0, False), (0, 2051, 64, 64, 3, True), (40, 512, 64, 64, 0, False), (0, 64, 8, 0, 2, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_prepare_on_both_sides_of_the_line(tokens, q_rank, rank, rot, dims, heads, halves, dtype):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(tokens + rank)
    head, plain, page, eps = rot + 5, 5, 4, 1e-5
    kv_off = q_rank + heads * head
    down = torch.randn(tokens, kv_off + rank + rot, generator=g).to(dtype)
    wq, wkv = ((1 + 0.1 * torch.randn(n, generator=g)).to(dtype) for n in (max(q_rank, 1), rank))
    freq = torch.rand(max(dims // 2, 1), generator=g)[: dims // 2]
    positions = torch.randint(0, 60, (tokens,), generator=g).int()
    table = torch.arange(1, tokens + 1).int().view(tokens, 1).repeat(1, 15)          # a page for each token, the last token's the sentinel
    table[-1] = 0 if tokens > 1 else 1
    plane = torch.full((tokens + 1, 1, page, rank + rot), 7.0, dtype=dtype, device="cuda")
    cq = torch.empty(tokens, q_rank, dtype=dtype, device="cuda") if q_rank else None
    rows = torch.full((tokens, heads * (rank + rot)), 7.0, dtype=dtype, device="cuda") if heads else None
    ops.latent_prepare(down.cuda(), q_rank, rank, rot, dims, wq.cuda() if q_rank else None, wkv.cuda(), eps, positions.cuda(), freq.cuda(), cq, torch.arange(tokens).int().cuda(), table.cuda(),
                       plane, page, kv_off=kv_off, halves=halves, queries=(rows, heads, head, plain) if heads else None)
    x, ang = down.double(), positions.double()[:, None] * freq.double()

    def turned(u):
        v, (a, b) = u.clone(), (slice(0, dims // 2), slice(dims // 2, dims)) if halves else (slice(0, dims, 2), slice(1, dims, 2))
        v[:, a], v[:, b] = u[:, a] * ang.cos() - u[:, b] * ang.sin(), u[:, b] * ang.cos() + u[:, a] * ang.sin()
        return v

    norm = lambda u, w: u / torch.sqrt(u.pow(2).mean(-1, keepdim=True) + eps) * w.double()
    # one rounding of the result; before it 32-bit sums, and angles of up to 60 radians, off by half a unit of 2^-18
    tol = dict(rtol=2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -18, atol=2.0 ** -15)
    if q_rank:
        torch.testing.assert_close(cq.cpu().double(), norm(x[:, :q_rank], wq), **tol)
    want = torch.full(plane.shape, 7.0, dtype=torch.float64)
    written = torch.cat((norm(x[:, kv_off: kv_off + rank], wkv), turned(x[:, kv_off + rank:])), 1)
    for t in range(tokens):
        if int(table[t, 0]):
            want[int(table[t, 0]), 0, int(positions[t]) % page] = written[t]
    torch.testing.assert_close(plane.cpu().double(), want, **tol)
    for h in range(heads):
        got = rows[:, h * (rank + rot): (h + 1) * (rank + rot)].cpu().double()
        torch.testing.assert_close(got[:, rank:], turned(x[:, h * head + plain: h * head + plain + rot]), **tol)
        assert bool((got[:, :rank] == 7.0).all())
