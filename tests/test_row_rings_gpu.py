"""Products of few rows through rings of slabs in shared memory, against float64 products of the same bfloat16 values: the edges of the blocks (rows of x 1, 8, 9, 16, 17, 32,
33 and 64; outputs that end inside a request of eight rows; fewer slabs of K than waves, and more than a ring holds), every shape that is built, ranges of K, the gates."""
from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from torchlet_amd.kernels import ops
    return ops


def _operands(M, N, K, seed, lead=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(torch.bfloat16).cuda()
    if lead:                                   # rows of a wider matrix
        wide = torch.full((M, K + lead), float("nan"), dtype=torch.bfloat16, device="cuda")
        wide[:, 8: 8 + K] = x
        x = wide[:, 8: 8 + K]
    return x, w


def _tol32(ref, K):
    # 32-bit sums of K products of exact bfloat16 operands: eight roundings of the running sum's size are not reached by a random walk of K of them
    return dict(rtol=2e-5, atol=8 * 2 ** -24 * math.sqrt(K) * float(ref.pow(2).mean().sqrt()))


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(1, 64), (7, 192), (50, 2112), (2050, 320), (4611, 128)])
def test_rings_as_the_library_deals_them(ops, M, N, K):
    x, w = _operands(M, N, K, M * 7 + N, lead=24)
    b = torch.randn(N, generator=torch.Generator().manual_seed(3)).cuda()
    ref = x.double() @ w.double().T
    out = torch.full((M + 1, N + 5), 3.0, device="cuda")
    ops.linear_ring_variant(x, w, b, out[:M, :N])
    torch.testing.assert_close(out[:M, :N].double(), ref + b.double(), **_tol32(ref, K))
    assert bool((out[:M, N:] == 3.0).all()) and bool((out[M] == 3.0).all())
    half = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    ops.linear(x, w, None, half)               # (the library's choice at these sizes)
    torch.testing.assert_close(half.double(), ref, rtol=2 ** -8, atol=_tol32(ref, K)["atol"])
    whole = torch.empty(M, N, device="cuda")
    ops.linear_ring_variant(x, w, None, whole)
    assert torch.equal(whole.bfloat16(), half)


@pytest.mark.parametrize("M", [3, 16, 30, 64])
@pytest.mark.parametrize("requests,rows", [(1, 8), (1, 5), (2, 16), (2, 9), (3, 24), (3, 17), (4, 30), (6, 48), (6, 41), (8, 64), (8, 50)])
def test_every_shape_of_the_rings(ops, M, requests, rows):
    N, K = 203, 1216                           # nineteen slabs: the waves have four or five each
    x, w = _operands(M, N, K, requests * 100 + rows + M)
    ref = x.double() @ w.double().T
    out = torch.full((M, N + 3), float("nan"), device="cuda")
    ops.linear_ring_variant(x, w, None, out[:, :N], requests, rows)
    torch.testing.assert_close(out[:, :N].double(), ref, **_tol32(ref, K))
    assert bool(out[:, N:].isnan().all())
    slabs = torch.full((3, M, N), float("nan"), device="cuda")
    ops.linear_ring_variant(x, w, None, slabs, requests, rows, parts=3)
    torch.testing.assert_close(slabs.double().sum(0), ref, **_tol32(ref, K))
    with pytest.raises(ops.KernelError, match="do not fit"):
        ops.linear_ring_variant(x, w, None, out[:, :N], requests, 8 * requests + 1)


@pytest.mark.parametrize("activation", ["silu", "relu", "gelu_tanh"])
@pytest.mark.parametrize("M,I,requests,rows", [(1, 40, 2, 8), (8, 100, 2, 7), (16, 75, 4, 16), (9, 75, 4, 11), (32, 130, 6, 24), (17, 130, 6, 21), (33, 97, 8, 32), (64, 97, 8, 29), (5, 300, 0, 0)])
def test_gates_in_the_rings(ops, activation, M, I, requests, rows):
    K = 576
    g = torch.Generator().manual_seed(I + M)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    gate, up = ((torch.randn(I, K, generator=g) / math.sqrt(K)).to(torch.bfloat16).cuda() for _ in range(2))
    w = ops.interleave_gate_up(gate, up)
    z, u = x.double() @ gate.double().T, x.double() @ up.double().T
    act = {"silu": torch.nn.functional.silu, "relu": torch.relu, "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[activation]
    out = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.linear_ring_variant(x, w, None, out, requests, rows, activation=activation)
    torch.testing.assert_close(out.double(), act(z) * u, rtol=2 ** -8, atol=1e-4)
    whole = torch.empty_like(out)
    ops.linear_swiglu(x, w, whole, activation)
    torch.testing.assert_close(whole.double(), act(z) * u, rtol=2 ** -8, atol=1e-4)


@pytest.mark.parametrize("M", [1, 8, 16])
def test_infinities_and_nan_stay_in_their_rows_and_columns(ops, M):
    """A block that is not full reads on into its slab's other rows: what lies there reaches outputs that are not stored."""
    N, K = 43, 384
    x, w = _operands(M, N, K, 5)
    x[0, 7], w[N - 1, 100], w[3, 0] = float("inf"), float("nan"), float("-inf")
    ref = x.float() @ w.float().T
    for requests, rows in ((1, 8), (3, 24), (6, 43), (0, 0)):
        out = torch.zeros(M, N, device="cuda")
        ops.linear_ring_variant(x, w, None, out, requests, rows)
        assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
