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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hidden", [4, 1028, 2048, 2050, 4096])
@pytest.mark.parametrize("slabs", [None, 0, 1, 2, 3, 4, 6, 8])
def test_a_tokens_sum_and_mixes_do_not_hang_on_the_steps_size(dtype, hidden, slabs):
    """The same tokens in steps of 40, of 256 and, on another kernel, of 257: the same bits."""
    g = torch.Generator(device="cuda").manual_seed(hidden + 1)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    T, own = 257, 40
    res, w, mu, state = rand(T, hidden), rand(hidden), torch.rand(5, hidden, generator=g, device="cuda"), rand(3, hidden)
    branch = None if slabs is None else rand(T, hidden).to(dtype) if slabs == 0 else rand(slabs, T, hidden)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    for post in (w, None):
        seen = {}
        for n in (own, 256, T):
            lens = [own - 1, n - own + 1]
            part = None if branch is None else branch[:n] if slabs == 0 else branch[:, :n].contiguous()
            mixes = torch.full((5, n, hidden), float("nan"), dtype=dtype, device="cuda")
            got = ops.settle_shift(res[:n].clone(), part, post, 1e-6, state, 0, i32([2, 1]), i32([0, lens[0], n]), i32([0] * lens[0] + [1] * lens[1]), mu, mixes)
            seen[n] = got[:own].clone(), mixes[:, :own].clone()
        for n in (own, 256):
            assert torch.equal(seen[n][0], seen[T][0]) and torch.equal(seen[n][1], seen[T][1]), n
