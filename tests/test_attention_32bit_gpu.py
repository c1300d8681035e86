"""The 32-bit attention kernel on the matrix cores: against the general kernel and 64 bits where a chunk, a page, a window or the written keys end."""
import math

import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,hd", [(7, 1, 16), (28, 4, 128), (4, 4, 112), (34, 2, 64), (2, 1, 256)])
@pytest.mark.parametrize("page", [4, 12, 16, 64])
@pytest.mark.parametrize("window,splits", [(0, 1), (0, 5), (33, 1), (17, 3)])
def test_against_the_general_kernel_and_64_bits(nh, nkv, hd, page, window, splits):
    g = torch.Generator().manual_seed(hd + page + window)
    lens, ctxs = [1, 17, 1, 1, 35], [63, 30, 64, 0, 0]                # the last key at the end of a chunk, behind it, and the only one
    totals = [a + b for a, b in zip(lens, ctxs)]
    R, T, width = len(lens), sum(lens), max(totals) // page + 2
    table = (torch.randperm(R * width, generator=g) + 1).view(R, width).int()
    kp = torch.full((R * width + 1, nkv, page, hd), math.nan)         # what no key has been written to yet may be anything
    vp = torch.full((R * width + 1, nkv, hd, page), math.nan)
    q = torch.randn(T, nh * hd, generator=g)
    ks, vs = ([torch.randn(n, nkv, hd, generator=g) for n in totals] for _ in range(2))
    for r, n in enumerate(totals):
        for p in range(n):
            kp[table[r, p // page], :, p % page] = ks[r][p]
            vp[table[r, p // page], :, :, p % page] = vs[r][p]
    starts = [sum(lens[:r]) for r in range(R + 1)]
    tq = ops.attention_tile_tokens(nh, nkv)
    tiles = [(r, t) for r, n in enumerate(lens) for t in range(0, n, tq)]
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), dev(starts), dev(ctxs), dev([r for r, _ in tiles]), dev([t for _, t in tiles]))
    out = {}
    for general in (False, True):
        out[general] = torch.full((T, nh * hd), math.nan, device="cuda")
        ops.paged_attention(args[0], out[general], *args[1:], len(tiles), tq, nh, nkv, hd, page, window, hd ** -0.5, splits, general=general)
    errors = {True: 0.0, False: 0.0}
    for r in range(R):
        k, v = (t.double().repeat_interleave(nh // nkv, 1) for t in (ks[r], vs[r]))
        at, keys = ctxs[r] + torch.arange(lens[r])[:, None], torch.arange(totals[r])[None, :]
        s = (q[starts[r]: starts[r + 1]].double().view(-1, nh, hd).transpose(0, 1) @ k.permute(1, 2, 0)) * hd ** -0.5
        s = s.masked_fill((keys > at) | ((keys <= at - window) if window else False), -math.inf)
        want = (torch.softmax(s, -1) @ v.transpose(0, 1)).transpose(0, 1).reshape(lens[r], nh * hd)
        for general in out:
            got = out[general][starts[r]: starts[r + 1]].cpu().double()
            # scores: hd products of order one in 32 bits, each rounded by 2^-24 of a sum of order sqrt(hd); their error moves every weight as much
            torch.testing.assert_close(got, want, rtol=1e-5, atol=2 ** -24 * math.sqrt(hd) * 8)
            errors[general] = max(errors[general], float((got - want).norm() / want.norm()))
    assert errors[False] <= 2 * errors[True] + 1e-7
