"""32-bit products of few rows through rings in shared memory: rounding of short sums, the same bits for a row whatever stands beside it, and nothing beyond the outputs; every shape that is built, for the
plain product, the gate and the rotation."""
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


# requests of eight weight rows and outputs (pairs) of a work-group: full, and with a last request or block that is not
PLAIN = [(1, 8), (1, 5), (2, 16), (2, 11), (3, 24), (3, 17), (4, 32), (4, 29), (6, 48), (6, 35), (8, 64), (8, 57)]
PAIRS = [(2, 8), (2, 5), (3, 12), (3, 9), (4, 16), (4, 14), (6, 24), (6, 17), (8, 32), (8, 29)]
# columns of K: one slab for one wave; up to three requests a work-group has eight waves, else four: one slab, two, a ring's worth and more a wave, some a slab more than others; 1024 and 2048: eight slabs a
# wave, from where the work-groups begin elsewhere
DEPTHS = [32, 160, 288, 512, 1056, 1024, 1184, 2048]


def _moved(K, requests):
    """Whether a work-group's sums begin elsewhere than at the first slab, so that their order is the shape's own."""
    return K % 1024 == 0 and K // 32 // (8 if requests <= 3 else 4) >= 8


def _bound(x, w, b=None):
    """See above: of what a sum's magnitudes add up to."""
    size = x.double().abs() @ w.double().abs().T + (0.0 if b is None else b.double().abs())
    return (19 + x.shape[1] / 256) * 2.0 ** -24 * size


def _same(a, c, moved, slack):
    return bool(((a.double() - c.double()).abs() <= slack).all()) if moved else torch.equal(a, c)


@pytest.mark.parametrize("requests, rows", PLAIN)
@pytest.mark.parametrize("K", DEPTHS)
def test_every_shape(requests, rows, K):
    N = 131
    g = torch.Generator(device="cuda").manual_seed(K + rows)
    x, w, b = torch.randn(16, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda"), torch.randn(N, generator=g, device="cuda")
    want, bound = x.double() @ w.double().T + b.double(), _bound(x, w, b)
    plain = torch.empty(16, N, device="cuda")
    ops.linear_f32_variant(x, w, b, plain, RINGS, 1, 8)
    seen = {}
    for M in (16, 9, 8, 1):
        out = torch.full((M + 1, N + 3), float("nan"), device="cuda")
        ops.linear_f32_variant(x[:M], w, b, out[:M, :N], RINGS, requests, rows)
        assert bool(((out[:M, :N].double() - want[:M]).abs() <= bound[:M]).all())
        assert bool(torch.isnan(out[M:]).all()) and bool(torch.isnan(out[:, N:]).all())
        seen[M] = out[:M, :N]
        assert torch.equal(seen[M], seen[16][:M])
    assert _same(seen[16], plain, _moved(K, 1) or _moved(K, requests), 2 * bound)
    with pytest.raises(ops.KernelError, match="do not fit"):
        ops.linear_f32_variant(x, w, b, plain, RINGS, requests, 8 * requests + 1)


def _plain(x, w, b=None):
    """The product through the rings as the library deals them: bits that any shape leaves but where its sums begin elsewhere."""
    out = torch.empty(x.shape[0], w.shape[0], device="cuda")
    ops.linear_f32_variant(x, w, b, out, RINGS)
    return out


@pytest.mark.parametrize("requests, rows", PAIRS + [(-1, 0)])
@pytest.mark.parametrize("K", DEPTHS)
def test_gates_in_every_shape(requests, rows, K):
    I = 67
    g = torch.Generator(device="cuda").manual_seed(K + rows)
    x, w = torch.randn(16, K, generator=g, device="cuda"), torch.randn(2 * I, K, generator=g, device="cuda") / K ** 0.5
    both, gated = _plain(x, w), torch.empty(16, I, device="cuda")
    ops.swiglu(both, gated, "silu")
    # silu(a) b for a and b each off by two orders' roundings: silu is at most |a| and its slope at most 1.1
    off = 2 * _bound(x, w)
    slack = 1.1 * off[:, :I] * (both[:, I:].abs() + off[:, I:]) + both[:, :I].abs() * off[:, I:] + 4 * 2.0 ** -24 * gated.abs()
    seen = {}
    for M in (16, 9, 8, 1):
        out = torch.full((M + 1, I + 1), float("nan"), device="cuda")
        assert ops.linear_gate_stacked(x[:M], w, out[:M, :I], "silu", (requests, rows))
        assert bool(torch.isnan(out[M:]).all()) and bool(torch.isnan(out[:, I:]).all())
        seen[M] = out[:M, :I]
        assert torch.equal(seen[M], seen[16][:M])
    assert _same(seen[16], gated, K % 1024 == 0, slack)
    if requests > 0:
        with pytest.raises(ops.KernelError, match="do not fit"):
            ops.linear_gate_stacked(x, w, gated, "silu", (requests, 4 * requests + 1))


@pytest.mark.parametrize("requests, rows", PAIRS + [(-1, 0)])
@pytest.mark.parametrize("K", DEPTHS)
@pytest.mark.parametrize("heads, kv_heads, hd", [(2, 1, 34), (3, 2, 24)])         # pairs of a work-group on both sides of a head's end
def test_rotations_in_every_shape(requests, rows, K, heads, kv_heads, hd):
    page = 3
    g = torch.Generator(device="cuda").manual_seed(K + rows + hd)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    N = (heads + 2 * kv_heads) * hd
    x, w, b, freq = rand(16, K), rand(N, K) / K ** 0.5, rand(N), torch.rand(hd // 2, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    table = (torch.arange(16 * 14) + 1).view(16, 14).int().cuda()
    table[7] = 0                                              # a padding row: its keys and values are dropped
    positions, req = i32([(17 * m) % 40 for m in range(16)]), i32(list(range(16)))
    planes = lambda: (torch.full((16 * 14 + 1, kv_heads, page, hd), 7.0, device="cuda"), torch.full((16 * 14 + 1, kv_heads, hd, page), 7.0, device="cuda"))
    both, (wk, wv) = _plain(x, w, b), planes()
    turned = both.clone()
    ops.rope_cache_write(turned, heads, kv_heads, hd, heads + kv_heads, positions, freq, req, table, wk, wv, page)
    slack = 4 * float(_bound(x, w, b).max()) + 4 * 2.0 ** -24 * float(both.abs().max())         # two elements off by two orders' roundings, and the turn's own
    seen = {}
    for M in (16, 9, 8, 1):
        out, (k, v) = torch.full((M + 1, N + 4), float("nan"), device="cuda"), planes()
        assert ops.linear_rope_cache_write(x[:M], w, b, out[:M], heads, kv_heads, hd, positions[:M], freq, req[:M], table[:M], k, v, page, pairs=False, rings=(requests, rows))
        assert bool(torch.isnan(out[M:]).all()) and bool(torch.isnan(out[:, heads * hd:]).all())
        seen[M] = out[:M, : heads * hd], k, v
        own = 1 + 14 * M
        assert torch.equal(seen[M][0], seen[16][0][:M]) and all(torch.equal(seen[M][i][:own], seen[16][i][:own]) and bool((seen[M][i][own:] == 7.0).all()) for i in (1, 2))
    for a, c in zip(seen[16], (turned[:, : heads * hd], wk, wv)):
        assert _same(a, c, K % 1024 == 0, slack)
