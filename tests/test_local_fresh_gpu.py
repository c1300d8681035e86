"""Single tokens whose attention puts their keys and values into their pages: the bits of the write ahead and the attention behind it, and nothing written elsewhere."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, kv_heads, dim, vdim", [(16, 4, 128, 128), (2, 2, 64, 64), (40, 2, 192, 64), (4, 4, 96, 48)])
@pytest.mark.parametrize("page, chunk, window, keep", [(16, 0, 0, 0), (8, 64, 0, 0), (8, 0, 40, 4), (24, 0, 1030, 0)])
@pytest.mark.parametrize("contexts", [[0, 31, 32, 63, 64, 1023], [1500, 7], [3000]])
@pytest.mark.parametrize("room", [40, 1200])          # keys that the block table has room for beyond the longest: a table of few keys leaves the heads to themselves
def test_same_bits_as_with_a_write_ahead(heads, kv_heads, dim, vdim, page, chunk, window, keep, contexts, room):
    g = torch.Generator(device="cuda").manual_seed(dim + page + window)
    R, width = len(contexts), (max(contexts) + room) // page + 1
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda").bfloat16()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    k, v = rand(R * width + 1, kv_heads, page, dim), rand(R * width + 1, kv_heads, vdim, page)
    table = (torch.randperm(R * width, generator=torch.Generator().manual_seed(1)) + 1).view(R, width).int().cuda()
    table[-1] = 0                                        # the last row belongs to no request: what it would write is dropped
    contexts = contexts + [3]
    table = torch.cat((table, table[:1] * 0))
    if R == 1:
        table[0] = torch.arange(1, width + 1).int().cuda()
    T = R + 1
    for r, p in enumerate(contexts):                     # the token's own place holds what some request left there
        k[table[r, p // page].long(), :, p % page] = float("nan")
        v[table[r, p // page].long(), :, :, p % page] = float("nan")
    k[0], v[0] = 0.0, 0.0
    rows = rand(T, heads * dim + kv_heads * (dim + vdim) + 8)
    q, kn, vn = rows[:, : heads * dim], rows[:, heads * dim: heads * dim + kv_heads * dim], rows[:, heads * dim + kv_heads * dim: heads * dim + kv_heads * (dim + vdim)]
    lists = (i32(list(range(T + 1))), i32(contexts), i32(list(range(T))), i32([0] * T), T)
    out = {}
    for how in ("ahead", "fresh"):
        kp, vp, o = k.clone(), v.clone(), torch.full((T, heads * vdim), float("nan"), dtype=torch.bfloat16, device="cuda")
        if how == "ahead":
            ops.kv_cache_write(kn, vn, lists[2], lists[1], table, kp, vp, page)
        ops.local_attention(q, o, kp, vp, table, lists[2], lists[1], heads, kv_heads, dim, vdim, page, dim ** -0.5, 20.0, chunk, window, 0.7, tiles=lists, keep_first=keep,
                            **({"fresh": (kn, vn)} if how == "fresh" else {}))
        out[how] = (o, kp, vp)
    live = [r for r in range(T) if int(table[r].max()) > 0]
    assert torch.equal(out["ahead"][0][live], out["fresh"][0][live]) and bool(torch.isfinite(out["fresh"][0][live].float()).all())
    for a, b in zip(out["ahead"][1:], out["fresh"][1:]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
