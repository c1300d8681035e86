"""Attention over prompts in tiles of 128 rows: weights are taken from each step's own maximum, so the order in which large and small scores come must not matter."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["rising", "falling", "one high", "far below", "alternating"])
@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("window", [0, 100])
def test_scores_of_any_order(shape, sink, window):
    from torchlet_amd.kernels import ops
    H, G, dim, page, n = 24, 12, 128, 16, 600                   # (24 heads x 600 tokens: enough for tiles of 128 rows)
    g = torch.Generator().manual_seed(len(shape))
    # every query holds `size` in its first place, and a key's first place makes its score (in units of log 2, about) on top of small random ones
    level = {"rising": torch.arange(n) * 0.5, "falling": -torch.arange(n) * 0.5, "one high": 300.0 * (torch.arange(n) == 70), "far below": -400.0 * (torch.arange(n) >= 64),
             "alternating": 60.0 * (torch.arange(n) // 64 % 2)}[shape]
    k = torch.randn(n, G, dim, generator=g) * 0.3
    k[:, :, 0] = level[:, None] / 8
    q = torch.randn(n, H, dim, generator=g) * 0.3
    q[:, :, 0] = 8 * dim ** 0.5 * 0.6931
    v = torch.randn(n, G, dim, generator=g)
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    s = torch.randn(H, generator=g) * 5 if sink else None
    blocks = -(-n // page)
    pad = lambda x: torch.cat((x, x.new_zeros(blocks * page - n, G, dim))).view(blocks, page, G, dim).permute(0, 2, 1, 3)
    kp = torch.cat((torch.zeros(1, G, page, dim, dtype=torch.bfloat16), pad(k))).contiguous().cuda()
    vp = torch.cat((torch.zeros(1, G, dim, page, dtype=torch.bfloat16), pad(v).transpose(2, 3))).contiguous().cuda()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    at = list(range(0, n, 16))
    out = torch.full((n, H * dim), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.local_attention(q.view(n, -1).cuda(), out, kp, vp, i32([list(range(1, blocks + 1))]), None, None, H, G, dim, dim, page, dim ** -0.5, window=window,
                        tiles=(i32([0, n]), i32([0]), i32([0] * len(at)), i32(at), len(at)), sink=s.cuda() if sink else None)
    back = torch.arange(n)[:, None] - torch.arange(n)[None]
    hidden = (back < 0) | (back >= window) if window else back < 0
    for h in range(H):
        x = (q[:, h].double() @ k[:, h // 2].double().T * dim ** -0.5).masked_fill(hidden, float("-inf"))
        top = x.max(1, keepdim=True).values if not sink else x.max(1, keepdim=True).values.clamp(min=float(s[h]))
        w = torch.exp(x - top)
        want = w @ v[:, h // 2].double() / (w.sum(1, keepdim=True) + (torch.exp(s[h].double() - top) if sink else 0.0))
        # three roundings to bfloat16, 2^-9 each of the terms' sizes: the weights', their sum's (it is made of the rounded ones) and the output's; scores of up to
        # 600 powers of two in 32 bits, 600 * 2^-22 in the exponent
        size = w @ v[:, h // 2].double().abs() / w.sum(1, keepdim=True)
        off = (out[:, h * dim: (h + 1) * dim].cpu().double() - want).abs()
        assert bool((off <= (3 * 2.0 ** -9 + 2.0 ** -12) * size + 1e-6).all()), (h, float((off / size).max()))
