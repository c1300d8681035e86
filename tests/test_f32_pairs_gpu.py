"""32-bit products of few rows whose gate, or whose rotation and cache write, is done by the product's own kernel: the bits of the separate launches (within rounding where the sums begin
elsewhere), and nothing written beside."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu

SIZES = [(1, 4), (5, 100), (96, 96), (517, 1056), (600, 2048), (1030, 1024)]      # (outputs or heads' columns, K): multiply-adds, rings, rings that begin elsewhere (K a multiple of 1024)


def _close(a, b, x, w, exact):
    if exact:
        return torch.equal(a, b)
    # two orders of a sum of K products, each with at most 18 + K / 256 + 1 roundings in a row; the gate or the turn makes at most four times as much of it
    return bool(((a - b).abs() <= 8 * (19 + x.shape[1] / 256) * 2.0 ** -24 * (1 + b.abs()) * float((x.abs() @ w.abs().T).max())).all())


@pytest.mark.parametrize("M", [1, 2, 4, 7, 9, 16])
@pytest.mark.parametrize("I, K", SIZES)
@pytest.mark.parametrize("act", ["silu", "relu", "gelu_tanh"])
def test_gate(M, I, K, act):
    g = torch.Generator(device="cuda").manual_seed(M + I + K)
    x, w = torch.randn(M, K + 4, generator=g, device="cuda")[:, 4:], torch.randn(2 * I, K, generator=g, device="cuda") / K ** 0.5
    gu, want = torch.empty(M, 2 * I, device="cuda"), torch.empty(M, I, device="cuda")
    ops.linear(x, w, None, gu)
    ops.swiglu(gu, want, act)
    out = torch.full((M + 1, I + 1), float("nan"), device="cuda")
    done = ops.linear_gate_stacked(x, w, out[:M, :I], act)
    assert done == (M <= 8 or K % 32 == 0)
    if done:
        assert _close(out[:M, :I], want, x, w, K % 1024 != 0)
        assert bool(torch.isnan(out[M:]).all()) and bool(torch.isnan(out[:, I:]).all())


@pytest.mark.parametrize("M", [1, 3, 8, 13])
@pytest.mark.parametrize("heads, kv_heads, hd, K", [(3, 1, 32, 96), (2, 2, 2, 20), (4, 2, 96, 1056), (14, 2, 64, 1024), (5, 5, 130, 2080)])
@pytest.mark.parametrize("writes", [True, False])
@pytest.mark.parametrize("page", [16, 3])
def test_rotation_and_cache_write(M, heads, kv_heads, hd, K, writes, page):
    g = torch.Generator(device="cuda").manual_seed(M + hd + K)
    N = (heads + (2 * kv_heads if writes else 0)) * hd
    x, w, b = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda") / K ** 0.5, torch.randn(N, generator=g, device="cuda")
    freq = torch.rand(hd // 2, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    positions, req, table = i32([(17 * m) % 40 for m in range(M)]), i32(list(range(M))), (torch.randperm(M * 14, generator=torch.Generator().manual_seed(M)) + 1).view(M, 14).int().cuda()
    if M > 1:
        table[M - 1] = 0                      # a padding row: its keys and values are dropped
    seen = []
    for fused in (False, True):
        k = torch.full((M * 14 + 1, kv_heads, page, hd), 7.0, device="cuda")
        v = torch.full((M * 14 + 1, kv_heads, hd, page), 7.0, device="cuda")
        cache = (req, table, k, v, page) if writes else (None, None, None, None, 0)
        out = torch.full((M + 1, N + 4), float("nan"), device="cuda")
        if fused:
            assert ops.linear_rope_cache_write(x, w, b, out[:M], heads, kv_heads if writes else 0, hd, positions, freq, *cache, pairs=False) == (M <= 8 or K % 32 == 0)
            if M > 8 and K % 32:
                return
            assert bool(torch.isnan(out[M:]).all()) and bool(torch.isnan(out[:, heads * hd:]).all())
        else:
            ops.linear(x, w, b, out[:M, :N])
            ops.rope_cache_write(out[:M], heads, kv_heads if writes else 0, hd, heads + (kv_heads if writes else 0), positions, freq, *cache)
        seen.append((out[:M, : heads * hd], k, v))
    for a, c in zip(*seen):
        assert _close(c, a, x, w, K % 1024 != 0)
