"""Attention over tiles of one request that brings fewer tokens than the step has rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("new", [17, 31, 32])
def test_a_request_shorter_than_the_steps_rows_is_not_left_out(new):
    from torchlet_amd.kernels import ops
    H, G, dim, page, ctx, T = 384, 48, 64, 16, 20, 32      # (384 heads: 32 rows are work enough for tiles of 128 rows)
    g = torch.Generator().manual_seed(new)
    blocks = -(-(ctx + T) // page)
    k = torch.randn(1 + blocks, G, page, dim, generator=g).bfloat16().cuda()
    v = torch.randn(1 + blocks, G, dim, page, generator=g).bfloat16().cuda()
    q = torch.randn(T, H * dim, generator=g).bfloat16().cuda()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    table = i32([list(range(1, blocks + 1))])
    at = (None, None)
    out, want = (torch.full((T, H * dim), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    tiles = (i32([0, new]), i32([ctx]), i32([0] * -(-new // 16)), i32(list(range(0, new, 16))), -(-new // 16))
    ops.local_attention(q, out, k, v, table, *at, H, G, dim, dim, page, dim ** -0.5, tiles=tiles)
    ops.local_attention(q[:new], want[:new], k, v, table, i32([0] * new), i32(list(range(ctx, ctx + new))), H, G, dim, dim, page, dim ** -0.5)
    # (weights rounded to bfloat16 and one rounding of the result on one way, of the result alone on the other: three of 2^-9 each)
    assert float((out[:new].float() - want[:new].float()).norm()) <= 3 * 2.0 ** -9 * float(want[:new].float().norm())
    assert bool(torch.isnan(out[new:].float()).all())
