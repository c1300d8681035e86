"""The chunked recurrences where the host knows a step's portions only as a bound, and beside requests of few tokens."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pays(monkeypatch):
    """Chunks wherever the sizes allow them, whatever the estimates say."""
    from torchlet_amd.kernels import ops
    real = ops._chunk_scratch

    class Pays:
        @staticmethod
        def tl_chunks_pay(*_):
            return 1
    monkeypatch.setattr(ops, "_chunk_scratch", lambda lib, *a, **k: real(Pays, *a, **k))


class _Step:
    """The matrix memory or fixed decays over random numbers, requests of `lens` tokens in the first rows of a step of `rows`."""

    def __init__(self, memory, lens, rows=None, H=2, dim=64, vdim=128):
        self.memory, self.lens, self.H, self.dim, self.vdim = memory, lens, H, dim, vdim
        g = torch.Generator().manual_seed(sum(lens))
        T = rows or sum(lens)
        self.qkv = torch.randn(T, 2 * H * dim + H * vdim, generator=g).cuda()
        self.gates = (torch.randn(T, 2 * H, generator=g) + 1.0).cuda()
        self.decay = torch.tensor([0.97, 0.999])[:H].cuda()
        self.start = torch.randn(len(lens), H, dim * vdim + (dim + 1 if memory else 0), generator=g).cuda()
        self.slots = torch.arange(len(lens), dtype=torch.int32, device="cuda")
        self.indptr = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")

    def run(self, qkv=None, gates=None, start=None, slots=None, indptr=None, **more):
        from torchlet_amd.kernels import ops
        qkv, gates = (self.qkv if qkv is None else qkv), (self.gates if gates is None else gates)
        state = (self.start if start is None else start).clone()
        slots, indptr = (self.slots if slots is None else slots), (self.indptr if indptr is None else indptr)
        out = torch.full((qkv.shape[0], self.H * self.vdim), float("nan"), device="cuda")
        H, dim, vdim = self.H, self.dim, self.vdim
        if self.memory:
            ops.mlstm_scan(qkv, H * dim, 2 * H * dim, gates, state, slots, indptr, out, H, dim, vdim, 9.0, dim ** -0.5, 1e-6, **more)
        else:
            ops.decay_scan(qkv, self.decay, state.view(state.shape[0], -1), slots, indptr, out, H, dim, vdim, **more)
        return out, state

    def alone(self, r):
        """Request r's tokens and nothing else in the step, and its own length given."""
        rows = slice(int(self.indptr[r]), int(self.indptr[r + 1]))
        n = self.lens[r]
        return self.run(self.qkv[rows].contiguous(), self.gates[rows].contiguous(), self.start[r: r + 1], self.slots[:1],
                        torch.tensor([0, n], dtype=torch.int32, device="cuda"), max_new_tokens=n)


@pytest.mark.parametrize("memory", [True, False])
@pytest.mark.parametrize("lens, rows, most", [([20], 20, 300), ([20], 400, None), ([31], 31, 32), ([40], 400, None)])
def test_a_request_shorter_than_the_bound_is_not_left_out(monkeypatch, memory, lens, rows, most):
    _pays(monkeypatch)
    step = _Step(memory, lens, rows)
    out, state = step.run(max_new_tokens=most)
    want, left = step.alone(0)
    assert torch.equal(out[: lens[0]], want) and torch.equal(state, left)
    assert bool(torch.isnan(out[lens[0]:]).all())


@pytest.mark.parametrize("memory", [True, False])
@pytest.mark.parametrize("most", [1, 40, 64, 1000])
def test_a_request_longer_than_was_said_is_taken_whole(monkeypatch, memory, most):
    _pays(monkeypatch)
    step = _Step(memory, [150, 3])
    out, state = step.run(max_new_tokens=most)
    for r, rows in enumerate((slice(0, 150), slice(150, 153))):
        want, left = step.alone(r)
        # (by the loop or by the chunks: 150 terms of like size, each rounding at most 2^-24 of a partial sum, on either way; the memory's outputs are quotients, whose
        # denominators may be small: its states show that every token was taken)
        assert float((state[r] - left[0]).norm()) <= 300 * 2.0 ** -24 * float(left.norm()) and bool(torch.isfinite(out[rows]).all())
        if not memory:
            assert float((out[rows] - want).norm()) <= 300 * 2.0 ** -24 * float(want.norm())


@pytest.mark.parametrize("memory", [True, False])
@pytest.mark.parametrize("where", ["query", "key", "value", "input gate"])
@pytest.mark.parametrize("token", [0, 5, 40, 63, 64, 100])
def test_infinities_and_nans_do_not_reach_the_tokens_before_them(monkeypatch, memory, where, token):
    from torchlet_amd.kernels import ops
    if where == "input gate" and not memory:
        pytest.skip("fixed decays have no gates")
    _pays(monkeypatch)
    step = _Step(memory, [130])
    clean, _ = step.run(max_new_tokens=130)
    H, dim = step.H, step.dim
    for bad in (float("inf"), float("nan")):
        qkv, gates = step.qkv.clone(), step.gates.clone()
        if where == "input gate":
            gates[token, 1] = float("nan")
        else:
            qkv[token, {"query": 3, "key": H * dim + 3, "value": 2 * H * dim + 3}[where]] = bad
        got, _ = step.run(qkv, gates, max_new_tokens=130)
        # (a chunk with such a value adds its tokens up in another order: 130 terms of like size, each rounding at most 2^-24 of a partial sum)
        assert float((got[:token] - clean[:token]).norm()) <= 130 * 2.0 ** -24 * float(clean[:token].norm()), bad
        assert not bool(torch.isfinite(got[token]).all()), bad
        monkeypatch.setattr(ops, "CHUNKED_FROM", 1 << 30)
        loop, _ = step.run(qkv, gates, max_new_tokens=130)
        monkeypatch.setattr(ops, "CHUNKED_FROM", 32)
        assert torch.equal(torch.isfinite(got), torch.isfinite(loop)), bad


def _portions(lens):
    from torchlet_amd.kernels import ops
    return ops.Portions.of(lens, ops.CHUNKED_FROM)


@pytest.mark.parametrize("memory", [True, False])
@pytest.mark.parametrize("lens", [[65, 0], [0, 0, 130, 0], [4] * 40, [1] * 9 + [65] + [31], [200, 33, 1, 64], [5, 1]])
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("passes", [True, False])
def test_every_request_moves_as_it_does_alone(monkeypatch, memory, lens, exact, passes):
    """With the lengths given and without, empty requests and decoded tokens beside long portions, in one pass over the chunks and in several."""
    from torchlet_amd.kernels import ops
    _pays(monkeypatch)
    step = _Step(memory, lens)
    want = {r: step.alone(r) for r, n in enumerate(lens) if n}
    if passes:                                         # (room for one chunk of every portion)
        per_chunk = step.H * (step.dim * step.vdim + (step.dim if memory else 0) + 1)
        monkeypatch.setattr(ops, "CHUNK_SCRATCH", per_chunk * max(1, sum(n >= 32 for n in lens) if exact else len(lens)))
    out, state = step.run(**({"portions": _portions(lens), "max_new_tokens": max(lens)} if exact else {}))
    at = 0
    for r, n in enumerate(lens):
        if n:
            assert torch.equal(out[at: at + n], want[r][0]) and torch.equal(state[r], want[r][1][0]), r
        else:
            assert torch.equal(state[r], step.start[r]), r
        at += n
