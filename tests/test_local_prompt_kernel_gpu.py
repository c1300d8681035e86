"""Attention over a paged cache for long portions of prompts (tiles of 128 rows) and for decoded tokens (heads together, keys split) against the kernel that walks the keys of one token and head.

Both get the same bfloat16 queries, keys and values.  The tiles round a weight to bfloat16 (half a unit: 2^-9 of it) and sum the rounded ones, so a
column moves by at most 2^-8 of the weights' mean of |value| (which the largest |value| bounds), and both round what they store (2^-9 of it each);
the factor 1.5 holds the 32-bit sums and the hardware's powers of two."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu
TILE = 16


def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


def _both(H, G, dim, vdim, page, ctx, new, g, window=0, chunk=0, pool=0, keep=0, cap=0.0, sink=None, turn=None, gated=False, spread=1.0, gain=1.0):
    R, lengths = len(ctx), [c + n for c, n in zip(ctx, new)]
    T = sum(new)
    draw = lambda *s: torch.randn(*s, generator=g, device="cuda")
    blocks = [-(-n // page) for n in lengths]
    width = max(blocks)
    pages = 1 + sum(blocks)
    k_plane = torch.full((pages, G, page, dim), float("nan"), dtype=torch.bfloat16, device="cuda")       # (slots that no token has written)
    v_plane = torch.full((pages, G, vdim, page), float("nan"), dtype=torch.bfloat16, device="cuda")
    order = torch.randperm(pages - 1, generator=g, device="cuda").tolist()
    table = torch.zeros((R, width), dtype=torch.int32)
    at = 0
    for r, n in enumerate(lengths):
        k, v = draw(n, G, dim) * spread, draw(n, G, vdim)
        first = max(0, ctx[r] - window + 1) if window else 0          # the first position that the portion reads
        if chunk:
            first = max(first, ctx[r] // chunk * chunk)
        for b in range(blocks[r]):
            held = (b + 1) * page > first or b * page < keep
            if not held:
                continue                                              # (given back: the entry names page 0, which holds nothing)
            p = 1 + order[at + b]
            table[r, b] = p
            m = min(page, n - b * page)
            k_plane[p, :, :m] = k[b * page: b * page + m].transpose(0, 1).bfloat16()
            v_plane[p, :, :, :m] = v[b * page: b * page + m].permute(1, 2, 0).bfloat16()
        at += blocks[r]
    table = table.cuda()
    pooled = None
    if pool:
        pw = max(-(-(n // pool + 1) // page) for n in lengths)
        pk = draw(1 + R * pw, G, page, dim).mul(spread).bfloat16()
        pv = draw(1 + R * pw, G, vdim, page).bfloat16()
        pooled = (pk, pv, (1 + torch.randperm(R * pw, generator=g, device="cuda")).int().view(R, pw), pool)
    q = draw(T, H * dim).mul(spread).bfloat16()
    gate = draw(T, H).bfloat16() if gated else None
    indptr = [0]
    for n in new:
        indptr.append(indptr[-1] + n)
    token_req = _i32([r for r, n in enumerate(new) for _ in range(n)])
    positions = _i32([ctx[r] + i for r, n in enumerate(new) for i in range(n)])
    tiles = [(r, t) for r, n in enumerate(new) for t in range(0, n, TILE)]
    outs = []
    for how in ((_i32(indptr), _i32(ctx), _i32([r for r, _ in tiles]), _i32([t for _, t in tiles]), len(tiles)), None):
        out = torch.full((T, H * vdim + 8), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.local_attention(q, out[:, : H * vdim], k_plane, v_plane, table, token_req, positions, H, G, dim, vdim, page, dim ** -0.5, cap, chunk, window,
                            gain, tiles=how, sink=sink, pooled=pooled, keep_first=keep, turn_back=turn, gate=gate)
        assert bool((out[:, H * vdim:] == 7.0).all())
        outs.append(out[:, : H * vdim].float())
    top = max(float(torch.nan_to_num(v_plane.float()).abs().max()), float(pooled[1].float().abs().max()) if pooled else 0.0)
    return outs[0], outs[1], top * gain * (2.0 ** 0.5 if turn else 1.0)


def _close(a, b, top):
    assert bool(torch.isfinite(b).all())
    assert bool(((a - b).abs() <= 1.5 * 2.0 ** -8 * (top + b.abs())).all()), float((a - b).abs().max())


@pytest.mark.parametrize("H, G, dim, vdim", [(4, 4, 128, 128), (16, 2, 64, 64), (6, 1, 192, 128), (34, 2, 128, 128), (5, 1, 64, 64)])
@pytest.mark.parametrize("page", [8, 16, 128])
@pytest.mark.parametrize("form", ["plain", "window", "chunk", "kept", "pooled", "capped"])
def test_long_portions_against_the_token_kernel(H, G, dim, vdim, page, form):
    g = torch.Generator(device="cuda").manual_seed(H + page)
    more = {"plain": {}, "window": dict(window=45, sink=torch.linspace(-3, 8, H, device="cuda")), "chunk": dict(chunk=96, gain=0.7),
            "kept": dict(window=70, keep=21, gated=True), "pooled": dict(window=33, pool=4, sink=torch.zeros(H, device="cuda")),
            "capped": dict(cap=5.0, turn=(torch.rand(vdim // 4, generator=g, device="cuda"), vdim // 2, False))}[form]
    # a decoded token, portions on both sides of where the tiles' kernel starts, of a whole tile and of several, after nothing and after cached tokens;
    # often enough for the step to go there
    ctx, new = [150, 0, 0, 77, 64, 3, 300], [1, 31, 32, 33, 128, 17, 200]
    times = -(-12288 // (H * (sum(new) - len(new))))
    _close(*_both(H, G, dim, vdim, page, ctx * times, new * times, g, **more))
    _close(*_both(H, G, dim, vdim, page, [11], [-(-12288 // H) + 1], g, spread=2.0, **more))


@pytest.mark.parametrize("H, G, dim, vdim", [(4, 4, 128, 128), (16, 2, 64, 64), (6, 1, 192, 64), (34, 2, 128, 128), (5, 1, 64, 128), (20, 1, 192, 128)])
@pytest.mark.parametrize("page", [8, 24])
@pytest.mark.parametrize("form", ["plain", "window", "chunk", "kept", "pooled", "capped", "halves"])
@pytest.mark.parametrize("ctx", [[0], [700], [0, 1, 127, 128, 1500, 33], [40] * 70])
@pytest.mark.parametrize("splits", [None, 1, 5])
def test_decoded_tokens_with_their_heads_together_against_the_token_kernel(H, G, dim, vdim, page, form, ctx, splits, monkeypatch):
    if splits:
        monkeypatch.setattr(ops, "local_decode_splits", lambda *a: splits)
    g = torch.Generator(device="cuda").manual_seed(H + page)
    freq = torch.rand(vdim // 4, generator=g, device="cuda")
    more = {"plain": {}, "window": dict(window=450, sink=torch.linspace(-3, 8, H, device="cuda")), "chunk": dict(chunk=352, gain=0.7),
            "kept": dict(window=170, keep=21, gated=True), "pooled": dict(window=333, pool=4, sink=torch.zeros(H, device="cuda"), gated=True),
            "capped": dict(cap=5.0, turn=(freq, vdim // 2, False)), "halves": dict(turn=(freq, vdim // 2, True), window=300)}[form]
    _close(*_both(H, G, dim, vdim, page, ctx, [1] * len(ctx), g, **more))
