"""Products over heads for few rows, against the products in 64 bits: 32-bit sums of products that are exact (2^-24 of the sum of their sizes a term's place), a gate's
sigmoid in 32-bit, one rounding to bfloat16."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 15, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("heads, N, K", [(3, 20, 64), (2, 512, 128), (5, 128, 512), (1, 7, 576), (4, 16, 1024)])
@pytest.mark.parametrize("gated", [False, True])
def test_heads(rows, heads, N, K, gated):
    g = torch.Generator(device="cuda").manual_seed(rows + N)
    x = torch.randn(rows, heads * (K + 8), generator=g, device="cuda").bfloat16()           # (a head's columns with others between)
    w = torch.randn(heads, N, K, generator=g, device="cuda").bfloat16()
    wide = torch.full((rows, heads * (N + 4)), 3.0, dtype=torch.bfloat16, device="cuda")
    gate = torch.randn(rows, heads * (N + 4), generator=g, device="cuda").bfloat16() if gated else None
    ops.heads_linear(x, K + 8, w, wide, N + 4, gate=gate)
    for h in range(heads):
        a, b = x[:, h * (K + 8): h * (K + 8) + K].double(), w[h].double()
        want, size = a @ b.T, a.abs() @ b.abs().T
        if gated:
            s = torch.sigmoid(gate[:, h * (N + 4): h * (N + 4) + N].double())
            want, size = want * s, size * s
        got = wide[:, h * (N + 4): h * (N + 4) + N].double()
        assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -24 * size).all())
        assert bool((wide[:, h * (N + 4) + N: (h + 1) * (N + 4)] == 3.0).all())
