"""Convolution, delta rule, norm and gate of single tokens in one launch: what the three launches give."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, kv_heads, dim, vdim", [(1, 1, 64, 16), (3, 3, 64, 52), (4, 2, 64, 64), (16, 8, 128, 128), (4, 1, 128, 64), (12, 1, 64, 20), (5, 5, 128, 124)])
@pytest.mark.parametrize("lens", [[1], [1, 1, 1, 1, 1], [1, 0, 5, 2]])
def test_one_launch_gives_what_three_give(dtype, heads, kv_heads, dim, vdim, lens):
    g = torch.Generator(device="cuda").manual_seed(dim + vdim)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    T, R, V = sum(lens), len(lens), heads * vdim
    C = 2 * kv_heads * dim + V
    proj = rand(T, C + V + 4).to(dtype)[:, : C + V]
    conv, gates, a_log, dt_bias, norm = rand(C, 4) * 0.5, rand(T, 2 * heads), rand(heads) - 1.0, rand(heads), 1.0 + 0.1 * rand(vdim)
    off = heads * dim * vdim + 4
    start = rand(R + 2, off + 3 * C + 4)
    slots = torch.tensor(list(range(R, 0, -1)), dtype=torch.int32, device="cuda")
    indptr = torch.tensor([sum(lens[:r]) for r in range(R + 1)], dtype=torch.int32, device="cuda")
    token_req = torch.tensor([r for r, n in enumerate(lens) for _ in range(n)], dtype=torch.int32, device="cuda")
    state, made, qkv, o = start.clone(), gates.clone(), torch.empty(T, C, device="cuda"), torch.empty(T, V, device="cuda")
    want = torch.empty(T, V + 8, dtype=dtype, device="cuda")[:, :V]
    ops.delta_prepare(proj, conv, made, a_log, dt_bias, state, off, slots, indptr, token_req, qkv, heads, kv_heads, dim, vdim, 4, dim ** -0.5, 1e-6)
    ops.delta_scan(qkv, made, state, slots, indptr, o, heads, kv_heads, dim, vdim)
    ops.gated_head_norm(o, proj[:, C:], norm, 1e-5, want, heads, vdim, gate="silu", gain=0.7)
    again, raw, wide = start.clone(), gates.clone(), torch.full((T, V + 8), 9.0, dtype=dtype, device="cuda")
    assert ops.delta_token(proj, C, conv, raw, a_log, dt_bias, again, off, slots, indptr, norm, 1e-5, wide[:, :V], heads, kv_heads, dim, vdim, 4, dim ** -0.5, 1e-6, 0.7)
    # the same sums in the same order: a multiply-add that one of the kernels rounds once and the other twice is all that may differ, and a step's state carries it on
    torch.testing.assert_close(again, state, rtol=2 ** -19, atol=2 ** -19)
    torch.testing.assert_close(wide[:, :V].float(), want.float(), rtol=2 ** -7 if dtype == torch.bfloat16 else 1e-5, atol=1e-5)
    assert torch.equal(raw, gates) and bool((wide[:, V:] == 9.0).all()) and torch.equal(again[0], start[0]) and torch.equal(again[R + 1], start[R + 1])


def test_what_it_is_not_built_for_is_left_to_the_three():
    f = lambda *shape: torch.zeros(*shape, device="cuda")
    i = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    for heads, kv, dim, vdim, taps, shift in ((1, 1, 32, 16, 4, 0), (1, 1, 64, 12, 4, 0), (1, 1, 64, 132, 4, 0), (5, 1, 64, 64, 4, 0), (1, 1, 64, 16, 3, 0), (1, 1, 64, 16, 4, 1)):
        C = 2 * kv * dim + heads * vdim
        state = torch.full((1, heads * dim * vdim + 3 * C), 3.0, device="cuda")
        assert not ops.delta_token(f(1, C + heads * vdim + shift)[:, shift:], C, f(C, taps), f(1, 2 * heads), f(heads), f(heads), state, heads * dim * vdim, i(0), i(0, 1), f(vdim), 1e-5,
                                   f(1, heads * vdim), heads, kv, dim, vdim, taps, 1.0, 1e-6)
        assert bool((state == 3.0).all())
