"""Decays, recurrence, norm and gate of single tokens in one launch: what the three launches give."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, dim, vdim, rank", [(3, 4, 4, 1), (32, 64, 64, 64), (1, 36, 52, 7), (2, 128, 128, 1024), (3, 100, 20, 17), (2, 68, 124, 16)])
@pytest.mark.parametrize("lens", [[1], [1, 1, 1, 1, 1], [1, 0, 3, 1]])
def test_one_launch_gives_what_three_give(dtype, heads, dim, vdim, rank, lens):
    g = torch.Generator(device="cuda").manual_seed(dim + rank)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    T, R, K, V, width = sum(lens), len(lens), heads * dim, heads * vdim, 24
    proj = rand(T, 2 * K + 2 * V + 4).to(dtype)[:, : 2 * K + 2 * V]
    z, w2t, w0 = rand(T, rank), rand(rank, K) * rank ** -0.5, rand(K) - 1.0
    bonus, norm, rows = rand(K), 1.0 + 0.1 * rand(V), rand(T, width)
    off = K * vdim + 4
    start = rand(R + 2, off + width)
    slots = torch.tensor(list(range(R, 0, -1)), dtype=torch.int32, device="cuda")
    indptr = torch.tensor([sum(lens[:r]) for r in range(R + 1)], dtype=torch.int32, device="cuda")
    state, decay, o, want = start.clone(), torch.empty(T, K, device="cuda"), torch.empty(T, V, device="cuda"), torch.empty(T, V, dtype=dtype, device="cuda")
    ops.channel_decay(z, w2t, w0, decay)
    ops.wkv_scan(proj, K, 2 * K, decay, bonus, state, slots, indptr, o, heads, dim, vdim, last_rows=rows, tail_off=off)
    ops.gated_head_norm(o, proj[:, 2 * K + V:], norm, 1e-5, want, heads, vdim, gate="silu")
    again, got = start.clone(), torch.full_like(want, float("nan"))
    assert ops.wkv_token(proj, K, 2 * K, 2 * K + V, z, w2t, w0, bonus, again, slots, indptr, norm, 1e-5, got, heads, dim, vdim, rows, off)
    # the same sums in the same order: a multiply-add that one of the kernels rounds once and the other twice is all that may differ
    torch.testing.assert_close(again, state, rtol=2 ** -21, atol=2 ** -21)
    torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -7 if dtype == torch.bfloat16 else 2e-6, atol=2e-6)
    assert torch.equal(again[0], start[0]) and torch.equal(again[R + 1], start[R + 1])


def test_what_it_is_not_built_for_is_left_to_the_three():
    f = lambda *shape: torch.zeros(*shape, device="cuda")
    i = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    for dim, vdim, shift in ((132, 4, 0), (4, 132, 0), (6, 4, 0), (4, 6, 0), (4, 4, 1)):
        K, V = dim, vdim
        proj = f(1, 2 * K + 2 * V + shift)[:, shift:]
        state = torch.full((1, K * V + 4), 3.0, device="cuda")
        assert not ops.wkv_token(proj, K, 2 * K, 2 * K + V, f(1, 2), f(2, K), f(K), f(K), state, i(0), i(0, 1), f(V), 1e-5, f(1, V), 1, dim, vdim, f(1, 4), K * V)
        assert bool((state == 3.0).all())
