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


@pytest.mark.parametrize("M", [2, 16, 17, 33, 64])
@pytest.mark.parametrize("requests,rows", [(1, 8), (2, 15), (3, 24), (4, 29), (6, 48), (8, 64)])
@pytest.mark.parametrize("K", [2048, 6144])                     # (6144: work-groups that begin at odd slabs and wrap at twenty-four)
def test_orders_turned_by_the_work_group(ops, M, requests, rows, K):
    """Rows of weights a multiple of 4 KB apart: every work-group begins at a slab of its own."""
    N = 64 * 11 + 5
    x, w = _operands(M, N, K, requests * 10 + M)
    ref = x.double() @ w.double().T
    out = torch.full((M, N), float("nan"), device="cuda")
    ops.linear_ring_variant(x, w, None, out, requests, rows)
    torch.testing.assert_close(out.double(), ref, **_tol32(ref, K))
    if K == 6144:                                               # (ranges of 2048 columns: eight slabs a wave, the fewest that are turned)
        slabs = torch.full((3, M, N), float("nan"), device="cuda")
        ops.linear_ring_variant(x, w, None, slabs, requests, rows, parts=3)
        torch.testing.assert_close(slabs.double().sum(0), ref, **_tol32(ref, K))
    if requests % 2 == 0:
        I = 32 * 9 + 7
        gate = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device="cuda")
        gu = ops.interleave_gate_up(w[:I], w[I: 2 * I])
        ops.linear_ring_variant(x, gu, None, gate, requests, rows // 2, activation="silu")
        torch.testing.assert_close(gate.double(), torch.nn.functional.silu(ref[:, :I]) * ref[:, I: 2 * I], rtol=2 ** -8, atol=1e-4)


@pytest.mark.parametrize("kind,N,K", [("whole", 2816, 2048), ("whole", 16000, 2048), ("whole", 6144, 4096), ("whole", 4608, 3584), ("gate", 5632, 2048), ("gate", 8192, 4096), ("gate", 25000, 2048),
                                      ("gate", 5120, 1536), ("slabs", 2048, 8192), ("slabs", 3584, 3584), ("groups", 1500, 2048)])
def test_a_rows_sums_do_not_hang_on_how_many_rows_there_are(ops, kind, N, K):
    """The same row first among 1, 2, 8, 9 and 16: the same bits (slabs are asked for from two rows on)."""
    g = torch.Generator().manual_seed(N)
    x = torch.randn(16, K, generator=g).to(torch.bfloat16).cuda()
    w = torch.randn(*((3,) if kind == "groups" else ()), (N + 31) // 32 * 64 if kind == "gate" else N, K, device="cuda", dtype=torch.bfloat16) * 0.02
    first = []
    for M in (1, 2, 8, 9, 16):
        if kind == "slabs":
            if M > 1:
                first.append(ops.linear_partials(x[:M], w)[:, 0])
            continue
        out = torch.empty(M, 3 * N if kind == "groups" else N, dtype=torch.bfloat16 if kind == "gate" else torch.float32, device="cuda")
        if kind == "gate":
            ops.linear_swiglu(x[:M], w, out)
        elif kind == "groups":
            ops.linear_groups(x[:M].expand(3, M, K).contiguous(), w, out)
        else:
            ops.linear(x[:M], w, None, out)
        first.append(out[0])
    assert all(torch.equal(f, first[0]) for f in first)


# (2048 rows of K and more, in steps of 2048: orders turned by the work-group; 9216 and 16000 outputs: runs of several strips; 16384: sixteen waves along K in both)
@pytest.mark.parametrize("nh,nkv,hd,hidden", [(16, 1, 128, 2048), (16, 2, 128, 2048), (32, 8, 128, 4096), (64, 4, 128, 2048), (121, 2, 128, 2048), (120, 4, 128, 2048), (3, 1, 64, 6144)])
def test_projection_of_one_row_that_makes_its_norm_itself_in_turned_orders(ops, nh, nkv, hd, hidden):
    g = torch.Generator().manual_seed(nh + hidden)
    width = (nh + 2 * nkv) * hd
    res, pend = torch.randn(1, hidden, generator=g).cuda(), torch.randn(3, 1, hidden, generator=g).cuda()
    nw = (1 + 0.1 * torch.randn(hidden, generator=g)).to(torch.bfloat16).cuda()
    w = torch.randn(width, hidden, device="cuda", dtype=torch.bfloat16) / math.sqrt(hidden)
    inv_freq = (1.0 / (1e6 ** (torch.arange(0, hd, 2).float() / hd))).cuda()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    where = (i32([9]), inv_freq, i32([0]), i32([[1]]))
    planes = lambda: (torch.zeros(2, nkv, 16, hd, dtype=torch.bfloat16, device="cuda"), torch.zeros(2, nkv, hd, 16, dtype=torch.bfloat16, device="cuda"))
    r0, h = res.clone(), torch.empty(1, hidden, dtype=torch.bfloat16, device="cuda")
    ops.add_rmsnorm(r0, pend, nw, 1e-6, h)
    (k0, v0), (k1, v1) = planes(), planes()
    q0, q1 = (torch.empty(1, width, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    assert ops.linear_rope_cache_write(h, w, None, q0, nh, nkv, hd, *where, k0, v0, 16)
    rout = torch.full_like(res, float("nan"))
    assert ops.linear_rope_cache_write_normed(res, pend, nw, 1e-6, rout, w, None, q1, nh, nkv, hd, *where, k1, v1, 16)
    assert torch.equal(rout, r0) and torch.equal(q1[:, : nh * hd], q0[:, : nh * hd]) and torch.equal(k1, k0) and torch.equal(v1, v0)
    plain = torch.empty(1, width, dtype=torch.bfloat16, device="cuda")
    ops.linear(h, w, None, plain)                               # (the values are not turned: the product as it is)
    exact = h.double() @ w.double().T
    torch.testing.assert_close(v1[1, :, :, 9].reshape(-1).double(), exact[0, (nh + nkv) * hd:], rtol=2 ** -8, atol=1e-4)



@pytest.mark.parametrize("M", [1, 9, 17])
def test_rows_too_far_apart_for_the_rings_offsets(ops, M):
    N, K, apart = 130, 128, 1 << 24            # (the bytes between rows, by a tile's rows, are beyond 32 bits)
    x, w = _operands(M, N, K, M)
    wide = torch.zeros(M, apart, dtype=torch.bfloat16, device="cuda")
    wide[:, :K] = x
    ref = x.double() @ w.double().T
    out = torch.full((M, N), float("nan"), device="cuda")
    ops.linear(wide[:, :K], w, None, out)
    torch.testing.assert_close(out.double(), ref, **_tol32(ref, K))
