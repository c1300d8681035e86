"""The sum and mixes of few tokens: every kind of branch, tokens that open their request and tokens behind others, slots at any place, and the step's size at which another kernel takes over."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[1, 1, 1], [3, 1, 7], [200, 56], [1, 256]])
@pytest.mark.parametrize("hidden, off, count", [(4, 4, 5), (1028, 5, 5), (2048, 8, 2), (4096, 4, 5)])
@pytest.mark.parametrize("slabs", [None, 0, 1, 2, 3, 4, 6, 8])
def test_sum_and_mixes(lens, hidden, off, count, slabs):
    g = torch.Generator(device="cuda").manual_seed(hidden + sum(lens))
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    T, R = sum(lens), len(lens)
    res, w, mu, state = rand(T, hidden), rand(hidden), torch.rand(count, hidden, generator=g, device="cuda"), rand(R + 1, off + hidden + 4)
    branch = None if slabs is None else rand(T, hidden).bfloat16() if slabs == 0 else rand(slabs, T, hidden)
    y = None if slabs is None else branch.double() if slabs == 0 else branch.double().sum(0)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    starts = [sum(lens[:r]) for r in range(R + 1)]
    for post in (w, None):
        mixes = torch.full((count, T, hidden), float("nan"), dtype=torch.bfloat16, device="cuda")
        got = ops.settle_shift(res, branch, post, 1e-6, state, off, i32(list(range(R, 0, -1))), i32(starts), i32([r for r, n in enumerate(lens) for _ in range(n)]), mu, mixes)
        x = res.double()
        if y is not None:
            x = x + (y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-6) * w.double() if post is not None else y)
        before = torch.cat((x[:1], x[:-1]))
        for r in range(R):
            before[starts[r]] = state[R - r, off: off + hidden].double()
        torch.testing.assert_close(got.double(), x, rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(mixes.double(), x + (before - x) * mu.double()[:, None], rtol=2 ** -8, atol=2e-5)      # (one rounding to bfloat16)
