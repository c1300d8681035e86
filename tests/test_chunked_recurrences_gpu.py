"""The recurrences with one decay per head and token over long portions, which go through chunks of 64 tokens: against 64 bits and the token loop, at
the edges of a chunk and of its tiles, from states that hold something, beside short portions, over several passes of the scratch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _linear(q, k, v, decay, S):
    out = []
    for t in range(q.shape[0]):
        S = S * decay[:, None, None] + v[t][:, :, None] * k[t][:, None]
        out.append((S * q[t][:, None]).sum(-1))
    return torch.stack(out), S


def _memory(q, k, v, gi, gf, cap, S, n, m):
    i = cap * torch.tanh(gi / cap)
    f = torch.nn.functional.logsigmoid(cap * torch.tanh(gf / cap))
    out, size = [], []
    SA, nA = S.abs(), n.abs()                          # the same sums of the terms' sizes
    for t in range(q.shape[0]):
        new = torch.maximum(f[t] + m, i[t])
        keep, take = torch.exp(f[t] + m - new), torch.exp(i[t] - new)
        S = keep[:, None, None] * S + (take[:, None] * k[t])[:, :, None] * v[t][:, None]
        SA = keep[:, None, None] * SA + (take[:, None] * k[t].abs())[:, :, None] * v[t].abs()[:, None]
        n, nA, m = keep[:, None] * n + take[:, None] * k[t], keep[:, None] * nA + take[:, None] * k[t].abs(), new
        den = (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6)[:, None]
        out.append((S * q[t][:, :, None]).sum(1) / den)
        size.append((SA * q[t].abs()[:, :, None]).sum(1) / den + out[-1].abs() * (nA * q[t].abs()).sum(-1)[:, None] / den)
    return torch.stack(out), torch.stack(size), S, n, m


def _forced(monkeypatch, chunked, scratch=None):
    """Chunks from 32 tokens on whatever the estimates say, or never."""
    from torchlet_amd.kernels import ops
    real = ops._chunk_scratch

    class Pays:
        @staticmethod
        def tl_chunks_pay(*_):
            return 1
    monkeypatch.setattr(ops, "CHUNKED_FROM", 32 if chunked else 1 << 30)
    if scratch is not None:
        monkeypatch.setattr(ops, "CHUNK_SCRATCH", scratch)
    monkeypatch.setattr(ops, "_chunk_scratch", lambda lib, *a: real(Pays, *a))


LENGTHS = [[63, 64, 65], [32, 1, 31, 128], [129, 2, 200]]


@pytest.mark.parametrize("lens", LENGTHS)
@pytest.mark.parametrize("H, dim, vdim", [(3, 20, 72), (2, 64, 128), (1, 132, 260), (5, 4, 4)])
def test_fixed_decays_in_chunks(monkeypatch, lens, H, dim, vdim):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(sum(lens) + dim)
    T, R = sum(lens), len(lens)
    qkv = torch.randn(T, 2 * H * dim + H * vdim, generator=g)
    decay = torch.tensor([0.0, 1.0, 0.97, 0.999, 0.5][:H])
    start = torch.randn(R + 1, H * dim * vdim, generator=g)
    slots = list(range(R, 0, -1))
    indptr = [0] + torch.tensor(lens).cumsum(0).tolist()
    results = {}
    # (the scratch of the last: one or two chunks of every request at a time)
    for name, chunked, scratch in (("loop", False, None), ("chunks", True, None), ("passes", True, 2 * R * H * (dim * vdim + 1))):
        _forced(monkeypatch, chunked, scratch)
        state, out = start.clone().cuda(), torch.full((T, H * vdim), float("nan"), device="cuda")
        ops.decay_scan(qkv.cuda(), decay.cuda(), state, torch.tensor(slots, dtype=torch.int32).cuda(), torch.tensor(indptr, dtype=torch.int32).cuda(), out, H, dim, vdim,
                       max_new_tokens=max(lens))
        results[name] = (out.cpu().double(), state.cpu())
        monkeypatch.undo()
    for r, n in enumerate(lens):
        x = qkv[indptr[r]: indptr[r + 1]].double()
        q, k, v = x[:, : H * dim].view(n, H, dim), x[:, H * dim: 2 * H * dim].view(n, H, dim), x[:, 2 * H * dim:].view(n, H, vdim)
        want, S = _linear(q, k, v, decay.double(), start[slots[r]].double().view(H, vdim, dim))
        errors = {}
        for name, (out, state) in results.items():
            got, left = out[indptr[r]: indptr[r + 1]].view(n, H, vdim), state[slots[r]].double().view(H, vdim, dim)
            errors[name] = float((got - want).norm() / want.norm())
            # 32-bit sums of up to a few hundred terms of like size: each rounding at most 2^-24 of a partial sum
            assert errors[name] < 400 * 2.0 ** -24 and float((left - S).norm() / S.norm()) < 400 * 2.0 ** -24, (name, errors)
        assert max(errors["chunks"], errors["passes"]) < 1.5 * errors["loop"] + 2.0 ** -22, errors
        if n < 32:
            assert torch.equal(results["chunks"][0][indptr[r]: indptr[r + 1]], results["loop"][0][indptr[r]: indptr[r + 1]])
    assert all(torch.equal(state[0], start[0]) for _, state in results.values())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens", LENGTHS)
@pytest.mark.parametrize("H, dim, vdim", [(3, 20, 72), (2, 64, 128), (1, 132, 260)])
def test_the_matrix_memory_in_chunks(monkeypatch, dtype, lens, H, dim, vdim):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(sum(lens) + dim)
    T, R, W = sum(lens), len(lens), dim * vdim + dim + 1
    qkv = torch.randn(T, 2 * H * dim + H * vdim + 4, generator=g).to(dtype)
    gates = torch.randn(T, 2 * H, generator=g) * 2
    gates[:, H:] += 1.5
    start = torch.randn(R + 1, H, W, generator=g)
    slots = list(range(R, 0, -1))
    indptr = [0] + torch.tensor(lens).cumsum(0).tolist()
    results = {}
    for name, chunked, scratch in (("loop", False, None), ("chunks", True, None), ("passes", True, 2 * R * H * W)):
        _forced(monkeypatch, chunked, scratch)
        state, out = start.clone().cuda(), torch.full((T, H * vdim), float("nan"), device="cuda")
        ops.mlstm_scan(qkv.cuda(), H * dim, 2 * H * dim, gates.cuda(), state, torch.tensor(slots, dtype=torch.int32).cuda(),
                       torch.tensor(indptr, dtype=torch.int32).cuda(), out, H, dim, vdim, 9.0, dim ** -0.5, 1e-6)
        results[name] = (out.cpu().double(), state.cpu())
        monkeypatch.undo()
    for r, n in enumerate(lens):
        rows = slice(indptr[r], indptr[r + 1])
        x, s0 = qkv[rows].double(), start[slots[r]].double()
        q, k = x[:, : H * dim].view(n, H, dim) * dim ** -0.5, x[:, H * dim: 2 * H * dim].view(n, H, dim)
        v = x[:, 2 * H * dim: 2 * H * dim + H * vdim].view(n, H, vdim)
        want, size, S, nn, m = _memory(q, k, v, gates[rows, :H].double(), gates[rows, H:].double(), 9.0, s0[:, : dim * vdim].view(H, dim, vdim), s0[:, dim * vdim: -1], s0[:, -1])
        left = torch.cat((S.reshape(H, -1), nn, m[:, None]), 1)
        for name, (out, state) in results.items():
            # a numerator's and a denominator's sums: every term is multiplied by up to n decays and added up n + dim times, each to within 2^-24 of
            # the sum of the terms' sizes (and a decay is an exponential of sums, good to a few units of its last place)
            off = (out[rows].view(n, H, vdim) - want).abs()
            assert bool((off <= (8 * n + dim + 16) * 2.0 ** -24 * size + 1e-12).all()), (name, float((off / size).max() * 2.0 ** 24))
            torch.testing.assert_close(state[slots[r]].double(), left, rtol=1e-4, atol=1e-4)
    assert all(torch.equal(state[0], start[0]) for _, state in results.values())


@pytest.mark.parametrize("lens", [[1024, 63, 2050], [1025, 1023]])
def test_the_matrix_memory_over_several_rounds_of_its_gates(monkeypatch, lens):
    """A work-group takes 16 stretches of 64 tokens a round: whole rounds, one more token and one less, and a short request beside."""
    test_the_matrix_memory_in_chunks(monkeypatch, torch.float32, lens, 2, 20, 24)
