"""Norms of rows whose branch lies in every number of slabs, in rows that end within a piece's reach, for few rows and for more than a GPU has compute units."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 300])
@pytest.mark.parametrize("hidden", [4, 1020, 2048, 3584, 4100, 6144, 6148])
@pytest.mark.parametrize("slabs", [None, 0, 1, 2, 3, 4, 5, 7, 8, 11])
def test_norms_after_a_branch(rows, hidden, slabs):
    """Sums of up to 12 numbers of order one in 32 bits, a norm's sum of `hidden` squares, one rounding to bfloat16 (2^-9)."""
    g = torch.Generator(device="cuda").manual_seed(rows + hidden)
    x, w = torch.randn(rows, hidden, generator=g, device="cuda"), torch.randn(hidden, generator=g, device="cuda")
    post = torch.randn(hidden, generator=g, device="cuda")
    branch = None if slabs is None else torch.randn(rows, hidden, generator=g, device="cuda").bfloat16() if slabs == 0 else torch.randn(slabs, rows, hidden, generator=g, device="cuda")
    y = torch.zeros(rows, hidden, dtype=torch.float64, device="cuda") if branch is None else branch.double() if slabs == 0 else branch.double().sum(0)
    unit = lambda v: v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-6)
    close = lambda got, want, r: torch.testing.assert_close(got.double(), want, rtol=r, atol=r)
    for weight in (w, w.bfloat16()):
        r, out = x.clone(), torch.empty(rows, hidden, dtype=torch.bfloat16, device="cuda")
        ops.add_rmsnorm(r, branch, weight, 1e-6, out)
        close(r, x.double() + y, 1e-5)
        close(out, unit(x.double() + y) * weight.double(), 2 ** -8)
        r = x.clone()
        ops.scaled_add_rmsnorm(r, branch, 0.5, weight, 1e-6, out)
        close(r, unit(0.5 * x.double() + y) * weight.double(), 1e-5)
        close(out, unit(0.5 * x.double() + y) * weight.double(), 2 ** -8)
    for normed in (post, None):
        r = x.clone()
        ops.sandwich_norm(r, branch, normed, 1e-6, None, w, 1e-6, out, branch_gain=0.5)
        want = x.double() + (0.5 * (unit(y) * post.double() if normed is not None else y) if branch is not None else 0.0)
        close(r, want, 1e-5)
        close(out, unit(want) * w.double(), 2 ** -8)
