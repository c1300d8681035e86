"""The latents' norms, rotation and cache write on both sides of 512 tokens (below: a work-group for each of them), the attention at the sizes that have kernels of their own (latents of
a multiple of 64 numbers beside 0, 32 or 64 rotated ones) and at others, and the merges of parts, against plain 64-bit formulas."""
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


@pytest.mark.parametrize("rot", [0, 32, 64])
@pytest.mark.parametrize("tile_rows,new", [(16, 1), (32, 2), (64, 5)])
@pytest.mark.parametrize("splits", [1, 2, 3, 63, 64])
@pytest.mark.parametrize("sink,window", [(True, 0), (False, 45)])
def test_attention_over_latents_of_512_numbers(rot, tile_rows, new, splits, sink, window):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(rot + splits)
    heads, rank, page, ctx, scale = 16, 512, 8, [0, 31, 333], 0.05
    D, bl = rank + rot, 44
    plane = (torch.randn(1 + 3 * bl, 1, page, D, generator=g)).bfloat16()
    table = (1 + torch.randperm(3 * bl, generator=g)).int().view(3, bl)
    T, tq = 3 * new, ops.latent_tile_tokens(heads, tile_rows)
    q = torch.randn(T, heads * D, generator=g).bfloat16()
    sinks = torch.linspace(-2, 4, heads) if sink else None
    tiles = [(r, t) for r in range(3) for t in range(0, new, tq)]
    out = torch.empty(T, heads * rank, dtype=torch.bfloat16, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    ops.latent_attention(q.cuda(), out, plane.cuda(), table.cuda(), i32([0, new, 2 * new, 3 * new]), i32(ctx), i32([r for r, _ in tiles]), i32([t for _, t in tiles]), len(tiles), tq, heads, rank, rot,
                         page, scale, None if sinks is None else sinks.cuda(), splits, max_new_tokens=new, window=window)
    for r in range(3):
        for i in range(new):
            n = ctx[r] + i + 1
            keys = plane[table[r].long()].reshape(-1, D)[max(0, n - window) if window else 0: n].double()
            s = q[r * new + i].double().view(heads, D) @ keys.T * scale
            den = torch.cat((s, sinks.double()[:, None]), 1) if sink else s
            w = torch.exp(s - den.logsumexp(1, keepdim=True))
            # the weights go to the product in bfloat16 and the result is rounded once: 2^-8 (half a unit in the last of 8 binary places) each, of the sum of magnitudes
            bound = 2.0 ** -7 * (w @ keys[:, :rank].abs()) + 1e-4
            assert bool(((out[r * new + i].cpu().double().view(heads, rank) - w @ keys[:, :rank]).abs() <= bound).all())


@pytest.mark.parametrize("vdim", [64, 128])
@pytest.mark.parametrize("splits", [2, 3, 9, 32])
def test_merge_of_a_decoded_tokens_parts(vdim, splits, monkeypatch):
    from torchlet_amd.kernels import ops
    heads, kv, dim, page, ctx, scale = 4, 1, 64, 8, [600, 0, 75], 0.1
    monkeypatch.setattr(ops, "local_decode_splits", lambda *a: splits)
    g = torch.Generator().manual_seed(vdim + splits)
    bl = 80
    k, v = (torch.randn(1 + 3 * bl, kv, page, n, generator=g).bfloat16() for n in (dim, vdim))
    table = (1 + torch.randperm(3 * bl, generator=g)).int().view(3, bl)
    q = torch.randn(3, heads * dim, generator=g).bfloat16()
    sink = torch.linspace(-1, 5, heads)
    out = torch.empty(3, heads * vdim, dtype=torch.bfloat16, device="cuda")
    i32 = lambda t: torch.tensor(t, dtype=torch.int32, device="cuda")
    tiles = (i32([0, 1, 2, 3]), i32(ctx), i32([0, 1, 2]), i32([0, 0, 0]), 3)
    ops.local_attention(q.cuda(), out, k.cuda(), v.transpose(2, 3).contiguous().cuda(), table.cuda(), i32([0, 1, 2]), i32(ctx), heads, kv, dim, vdim, page, scale, tiles=tiles, sink=sink.cuda())
    for r in range(3):
        keys, values = (p[table[r].long()][:, 0].reshape(bl * page, -1)[: ctx[r] + 1].double() for p in (k, v))
        s = q[r].double().view(heads, dim) @ keys.T * scale
        w = torch.exp(s - torch.cat((s, sink.double()[:, None]), 1).logsumexp(1, keepdim=True))
        bound = 2.0 ** -7 * (w @ values.abs()) + 1e-4          # (as above)
        assert bool(((out[r].cpu().double().view(heads, vdim) - w @ values).abs() <= bound).all())


@pytest.mark.parametrize("rank", [64, 80, 128, 192, 256, 320, 384, 448, 512])        # (80: the kernel by sizes that come with the call)
@pytest.mark.parametrize("rot", [0, 32, 64, 96, 16])                                 # (as 96; with 16 only rows of whole pieces of 32, so 80 alone)
@pytest.mark.parametrize("tile_rows,new,splits", [(16, 1, 1), (16, 1, 3), (32, 2, 1), (64, 5, 1), (64, 5, 2)])
def test_attention_at_every_size_that_has_a_kernel(rank, rot, tile_rows, new, splits):
    from torchlet_amd.kernels import ops
    D = rank + rot
    if D % 32:
        return
    g = torch.Generator().manual_seed(D + splits)
    heads, page, ctx, scale, bl = 16, 8, [3, 77], 0.08, 12
    plane = torch.randn(1 + 2 * bl, 1, page, D, generator=g).bfloat16()
    table = (1 + torch.randperm(2 * bl, generator=g)).int().view(2, bl)
    T, tq = 2 * new, ops.latent_tile_tokens(heads, tile_rows)
    q = torch.randn(T, heads * D, generator=g).bfloat16()
    tiles = [(r, t) for r in range(2) for t in range(0, new, tq)]
    out = torch.empty(T, heads * rank, dtype=torch.bfloat16, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    ops.latent_attention(q.cuda(), out, plane.cuda(), table.cuda(), i32([0, new, 2 * new]), i32(ctx), i32([r for r, _ in tiles]), i32([t for _, t in tiles]), len(tiles), tq, heads, rank, rot,
                         page, scale, None, splits, max_new_tokens=new, window=0)
    for r in range(2):
        for i in range(new):
            keys = plane[table[r].long()].reshape(-1, D)[: ctx[r] + i + 1].double()
            w = torch.softmax(q[r * new + i].double().view(heads, D) @ keys.T * scale, 1)
            bound = 2.0 ** -7 * (w @ keys[:, :rank].abs()) + 1e-4          # (as above)
            assert bool(((out[r * new + i].cpu().double().view(heads, rank) - w @ keys[:, :rank]).abs() <= bound).all())
