"""32-bit products of few rows through rings in shared memory: rounding of short sums, the same bits for a row whatever stands beside it, and nothing beyond the outputs."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu

RINGS = 9


@pytest.mark.parametrize("N, K", [(1, 32), (7, 96), (300, 96), (257, 992), (2100, 1024), (513, 2080), (4100, 224), (33000, 64)])
@pytest.mark.parametrize("bias", [False, True])
def test_rows_by_themselves_and_together(N, K, bias):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    wide = torch.randn(16, K + 8, generator=g, device="cuda")
    x, w = wide[:, 4: K + 4], torch.randn(N, K, generator=g, device="cuda")
    b = torch.randn(N, generator=g, device="cuda") if bias else None
    want = x.double() @ w.double().T + (b.double() if bias else 0.0)
    # a sum of K products in 32 bits, at most K roundings in a row of what its magnitudes add up to; the longest row here is a pair of products, pairs of pairs, slabs of 32
    # columns dealt to eight sums: 8 + 2 + K / 256 + 8 roundings
    bound = (18 + K / 256 + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + (b.double().abs() if bias else 0.0))
    seen = {}
    for M in (16, 9, 8, 5, 1):
        out = torch.full((M + 1, N + 3), float("nan"), device="cuda")
        ops.linear_f32_variant(x[:M], w, b, out[:M, :N], RINGS)
        assert bool(((out[:M, :N].double() - want[:M]).abs() <= bound[:M]).all())
        assert bool(torch.isnan(out[M:]).all()) and bool(torch.isnan(out[:, N:]).all())
        seen[M] = out[:M, :N]
    for M in (9, 8, 5, 1):
        assert torch.equal(seen[M], seen[16][:M])
