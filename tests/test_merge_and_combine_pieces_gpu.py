"""Sums in pieces of 16 bytes: the weighted sum of the chosen experts' rows against the same sum of single numbers (equal to the bit: the order is the same), and
the merge of a split attention over latents against the attention that was not split (32-bit sums in another order, one rounding to bfloat16)."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [8, 12, 1024, 1032, 2048, 4100])
@pytest.mark.parametrize("top", [1, 3, 4, 6, 8, 9])
@pytest.mark.parametrize("identity, shared", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_combine(width, top, identity, shared, dtype):
    g = torch.Generator(device="cuda").manual_seed(width + top)
    T = 5
    draw = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    y, x, add = draw(T * top, width), draw(T, width), draw(T, width)
    w = torch.rand(T, top, generator=g, device="cuda")
    slots = torch.randperm(T * top, generator=g, device="cuda").int()
    offsets = torch.tensor([0, T * top // 2, T * top * 3 // 4], dtype=torch.int32, device="cuda")
    more = dict(identity=(x, offsets, 2) if identity else None, addend=add if shared else None)
    out = torch.empty(T, width, dtype=dtype, device="cuda")
    ops.combine(y, slots, w, out, **more)
    shifted = torch.empty(T * top * width + 1, dtype=dtype, device="cuda")[1:].view(T * top, width)      # (off 16 bytes: the kernel of single numbers)
    shifted.copy_(y)
    want = torch.empty_like(out)
    ops.combine(shifted, slots, w, want, **more)
    assert torch.equal(out, want)


@pytest.mark.parametrize("rank, rot", [(512, 64), (64, 0), (30, 2), (36, 4)])
@pytest.mark.parametrize("splits", [2, 7, 8, 9, 64])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_merge(rank, rot, splits, dtype):
    g = torch.Generator(device="cuda").manual_seed(rank + splits)
    heads, page, ctx = 3, 16, [700, 5]
    width = 44
    plane = torch.randn(1 + 2 * width, 1, page, rank + rot, generator=g, device="cuda").to(dtype)
    table = (1 + torch.arange(2 * width, device="cuda")).int().view(2, width)
    q = torch.randn(2, heads * (rank + rot), generator=g, device="cuda").to(dtype)
    outs = []
    for n in (1, splits):
        out = torch.empty(2, heads * rank, dtype=dtype, device="cuda")
        ops.latent_attention(q, out, plane, table, None, torch.tensor(ctx, dtype=torch.int32, device="cuda"), None, None, 2, 1, heads, rank, rot, page,
                             (rank + rot) ** -0.5, torch.zeros(heads, device="cuda"), n, max_new_tokens=1)
        outs.append(out.double())
    # weights and sums are 32-bit either way (bfloat16 weights on the matrix cores: half a unit of 2^-8 of each against another maximum), then one rounding
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -18
    assert bool(((outs[0] - outs[1]).abs() <= 2 * eps * (outs[0].abs() + float(plane.abs().max()))).all())
