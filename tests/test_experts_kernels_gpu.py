"""The products over the experts' rows, each kernel alone, at the sizes where one can go wrong: groups at the edges of its tiles, empty groups,
more groups than a wave has lanes, columns that end inside a tile or a 16-byte piece, slots of no group left alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ACTS = {"none": lambda z: z, "relu2": lambda z: torch.relu(z) ** 2, "silu": lambda z: z * torch.sigmoid(z),
        "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh"), "gelu": torch.nn.functional.gelu}


def _plain(x, src, w, offsets, act):
    """The product in 64 bits, and the sum of its terms' sizes."""
    rows = (x if src is None else x[src.long()]).double()
    y, size = [], []
    for g in range(w.shape[0]):
        r = rows[offsets[g]: offsets[g + 1]]
        y.append(r @ w[g].double().T)
        size.append(r.abs() @ w[g].double().abs().T)
    y, size = torch.cat(y), torch.cat(size)
    if act.endswith("_pairs"):
        f = ACTS[act[:-6]]
        return f(y[:, 0::2]) * y[:, 1::2], size[:, 0::2] * y[:, 1::2].abs() + size[:, 1::2] * f(y[:, 0::2]).abs() + 1e-6 * size[:, 0::2] * size[:, 1::2]
    return ACTS[act](y), size * (1 + 2 * y.abs() if act == "relu2" else 2)


@pytest.mark.parametrize("counts, N, K, act", [
    ([0, 1, 15, 16, 17, 0], 96, 64, "none"), ([63, 64, 65], 260, 192, "relu2"), ([127, 128, 129, 0, 1], 130, 128, "silu_pairs"),
    ([255, 256, 257], 512, 448, "gelu_tanh_pairs"), ([i * 7 % 23 for i in range(130)], 32, 64, "gelu"), ([3, 0, 2], 24, 1024, "relu2_pairs")])
@pytest.mark.parametrize("which", range(6))
def test_experts_kernels_at_their_edges(which, counts, N, K, act):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(N + K)
    S, tokens = sum(counts), 40
    offsets = [0] + torch.tensor(counts).cumsum(0).tolist()
    w = (torch.randn(len(counts), N, K, generator=g) / K ** 0.5).bfloat16()
    for routed in (True, False):
        x = torch.randn(tokens if routed else S + 3, K, generator=g).bfloat16()
        src = torch.randint(0, tokens, (S + 3,), generator=g, dtype=torch.int32) if routed else None
        cols = N // 2 if act.endswith("_pairs") else N
        out = torch.full((S + 3, cols), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.experts_linear_variant(x.cuda(), None if src is None else src.cuda(), w.cuda(), torch.tensor(offsets, dtype=torch.int32).cuda(), out, act, which)
        want, size = _plain(x, src, w, offsets, act)
        assert bool((out[S:] == 7.0).all())
        # one rounding to bfloat16 (2^-9 of the value), and sums of K products in 32 bits (each step at most 2^-24 of the terms' sizes)
        off = (out[:S].cpu().double() - want).abs()
        assert bool((off <= 2.0 ** -8 * want.abs() + (K + 8) * 2.0 ** -23 * size + 1e-9).all()), float((off - 2.0 ** -8 * want.abs()).max())


def test_the_dispatch_takes_every_size_a_call_may_have():
    """From one slot to thousands, K on both sides of the few-rows kernel's line: the dispatch's choice gives what the general kernel gives."""
    from torchlet_amd.kernels import ops
    g = torch.Generator(device="cuda").manual_seed(1)
    for G, N, K in ((4, 64, 128), (8, 256, 2176), (3, 40, 96)):
        w = (torch.randn(G, N, K, generator=g, device="cuda") / K ** 0.5).bfloat16()
        for S in (1, 7, 8 * G, 8 * G + 1, 40 * G, 200 * G):
            x = torch.randn(S, K, generator=g, device="cuda").bfloat16()
            counts = torch.bincount(torch.randint(0, G, (S,), generator=g, device="cuda"), minlength=G)
            offsets = torch.cat((torch.zeros(1, dtype=torch.long, device="cuda"), counts.cumsum(0))).int()
            got, want = torch.empty(S, N, dtype=torch.bfloat16, device="cuda"), torch.empty(S, N, dtype=torch.bfloat16, device="cuda")
            ops.experts_linear(x, None, w, offsets, got, "silu")
            ops.experts_linear(x, None, w, offsets, want, "silu", general=True)
            # both round sums of the same products once: at most neighbouring bfloat16 numbers, and near zero the sums' own error
            torch.testing.assert_close(got.float(), want.float(), rtol=2.0 ** -7, atol=4 * K * 2.0 ** -24)
