"""The 32-bit tile kernel's sizes of tiles give the same bits, and the elementwise activation in whole pieces those of the numbers one by one."""
import math

import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [17, 63, 64, 65, 129, 300])
@pytest.mark.parametrize("N, K", [(64, 4), (65, 36), (127, 64), (130, 100), (516, 252)])
@pytest.mark.parametrize("bias", [False, True])
def test_every_tile_gives_the_same_bits(M, N, K, bias):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda") / math.sqrt(K)
    b = torch.randn(N, generator=g, device="cuda") if bias else None
    out = {}
    for tile in (4, 5, 6):
        out[tile] = torch.full((M, N + 4), 7.0, device="cuda")
        ops.linear_f32_variant(x, w, b, out[tile][:, :N], tile)
        assert bool((out[tile][:, N:] == 7.0).all())
    by_rule = torch.empty(M, N, device="cuda")
    ops.linear(x, w, b, by_rule)
    assert torch.equal(out[4], out[5]) and torch.equal(out[4], out[6]) and torch.equal(out[4][:, :N], by_rule)
    want = x.double() @ w.double().T + (b.double() if bias else 0.0)
    torch.testing.assert_close(by_rule.double(), want, rtol=2e-5, atol=8 * 2 ** -24 * math.sqrt(K))


@pytest.mark.parametrize("n", [1, 7, 8, 2048, 2056, 2051, 256 * 8 * 3 + 8])
@pytest.mark.parametrize("kind", ["relu2", "silu", "gelu_tanh", "gelu"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_activation_in_pieces(n, kind, dtype):
    x = (torch.randn(n + 1, generator=torch.Generator().manual_seed(n)) * 2).to(dtype).cuda()
    pieces, single = x[:n].clone(), torch.cat((x[:1], x[:n])).clone()[1:]          # (the second one begins off a 16-byte boundary)
    ops.activation(pieces, kind)
    ops.activation(single, kind)
    assert torch.equal(pieces, single)


def test_more_rows_than_a_launch_has_of_the_smallest_tiles():
    M, N, K = 65535 * 64 + 3, 64, 4
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    out = torch.empty(M, N, device="cuda")
    ops.linear(x, w, None, out)
    for part in (slice(0, 130), slice(M - 130, M)):
        torch.testing.assert_close(out[part].double(), x[part].double() @ w.double().T, rtol=2e-5, atol=8 * 2 ** -24 * math.sqrt(K))


@pytest.mark.parametrize("M", [17, 31, 32, 33, 97, 130])
@pytest.mark.parametrize("N, K", [(31, 28), (33, 32), (64, 60), (100, 224), (130, 1028)])
def test_tiles_of_small_blocks_and_of_large_ones_give_the_same_bits(M, N, K):
    """One slab or none, a rest of a slab, more slabs than are in flight; rows of x wider than K, rows of the result wider than N."""
    g = torch.Generator(device="cuda").manual_seed(M * K + N)
    x, w = torch.randn(M, K + 8, generator=g, device="cuda")[:, :K], torch.randn(N, K, generator=g, device="cuda") / math.sqrt(K)
    out = {}
    for tile in (4, 5, 6, 7, 8):
        out[tile] = torch.full((M, N + 3), 7.0, device="cuda")
        ops.linear_f32_variant(x, w, None, out[tile][:, :N], tile)
        assert torch.equal(out[tile], out[4])
    assert bool((out[4][:, N:] == 7.0).all())
    torch.testing.assert_close(out[4][:, :N].double(), x.double() @ w.double().T, rtol=2e-5, atol=8 * 2 ** -24 * math.sqrt(K))


def test_what_lies_beyond_a_row_reaches_no_sum():
    """Columns past K, rows past M and N: infinities there leave every result finite."""
    M, N, K = 40, 40, 36
    x, w = torch.full((M + 1, K + 28), math.inf, device="cuda"), torch.full((N + 8, K), math.inf, device="cuda")
    x[:M, :K], w[:N] = 1.0, 2.0
    for tile in (4, 5, 6, 7, 8):
        out = torch.empty(M, N, device="cuda")
        ops.linear_f32_variant(x[:M, :K], w[:N], None, out, tile)
        assert torch.equal(out, torch.full_like(out, 2.0 * K))
