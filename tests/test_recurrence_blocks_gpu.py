"""Long portions of the delta rule and of the selective recurrence in blocks of 16 tokens, against the recurrences token by token in 64 bits."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _always(monkeypatch):
    """The small sizes of these tests go through the blocks as well, whatever the estimate says."""
    lib = ops._lib("recurrent")
    monkeypatch.setattr(lib, "tl_blocks_pay", lambda *sizes: 1)


def _inputs(kind, lens, H, G, dim, vdim, seed):
    g = torch.Generator().manual_seed(seed)
    T = sum(lens)

    def unit(x):
        return x / x.norm(dim=-1, keepdim=True)
    q, k = (unit(torch.randn(T, G, dim, generator=g)) for _ in "qk")
    v = torch.randn(T, H * vdim, generator=g)
    decay = 0.8 + 0.2 * torch.rand(T, H, generator=g)
    decay[torch.rand(T, H, generator=g) < 0.02] = 0.0            # a decay of zero forgets what was
    x = torch.cat((q.reshape(T, -1), k.reshape(T, -1), v), 1).contiguous()
    return x, torch.cat((torch.rand(T, H, generator=g), decay), 1).contiguous(), torch.randn(H, generator=g), torch.randn(len(lens), H * dim * vdim + 4, generator=g) * 0.3


def _plain(kind, x, gates, skip, state, lens, H, G, dim, vdim):
    x, gates, state = x.double(), gates.double(), state.double().clone()
    of, out, at = torch.arange(H) // (H // G), [], 0
    for r, n in enumerate(lens):
        S = state[r, : H * dim * vdim].view(H, vdim, dim).clone()
        for t in range(at, at + n):
            q, k = x[t, : G * dim].view(G, dim)[of], x[t, G * dim: 2 * G * dim].view(G, dim)[of]
            v, beta = x[t, 2 * G * dim:].view(H, vdim), gates[t, :H, None]
            S = S * gates[t, H:, None, None]
            u = beta * (v - (S * k[:, None]).sum(-1)) if kind == "delta" else beta * v
            S = S + u[:, :, None] * k[:, None]
            o = (S * q[:, None]).sum(-1)
            out.append((o if kind == "delta" else o + skip.double()[:, None] * v).reshape(-1))
        state[r, : H * dim * vdim] = S.reshape(-1)
        at += n
    return torch.stack(out), state


def _run(kind, x, gates, skip, state, lens, H, G, dim, vdim, **more):
    state = state.clone().cuda()
    out = torch.full((sum(lens), H * vdim), float("nan"), device="cuda")
    slots = torch.arange(len(lens), dtype=torch.int32, device="cuda")
    indptr = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    args = (x.cuda(), gates.cuda()) + ((skip.cuda(),) if kind == "selective" else ()) + (state, slots, indptr, out, H, G, dim, vdim)
    (ops.delta_scan if kind == "delta" else ops.selective_scan)(*args, **more)
    return out.cpu(), state.cpu()


# lengths: the fewest that go through blocks, one short of them, whole and broken blocks, single tokens and an empty request beside them; sizes: whole tiles, broken
# ones, every number of tiles a wave, rows that cannot be read in pieces (which stay with the token loop), and numbers of heads that are dealt out over the XCDs
@pytest.mark.parametrize("kind", ["delta", "selective"])
@pytest.mark.parametrize("H, G, dim, vdim", [(4, 2, 128, 128), (5, 1, 64, 40), (2, 2, 100, 36), (6, 1, 36, 20), (1, 1, 256, 24), (2, 1, 132, 16), (2, 1, 30, 17),
                                               (8, 4, 64, 40), (16, 8, 128, 36)])
@pytest.mark.parametrize("lens", [[128], [127], [1, 128, 0, 161, 15, 144], [259, 129]])
@pytest.mark.parametrize("exact", [True, False])
def test_blocks_against_the_recurrence(kind, H, G, dim, vdim, lens, exact):
    x, gates, skip, state = _inputs(kind, lens, H, G, dim, vdim, dim + len(lens))
    more = dict(portions=ops.Portions.of(lens, ops.BLOCKS_FROM)) if exact else {}
    out, after = _run(kind, x, gates, skip, state, lens, H, G, dim, vdim, **more)
    want, want_state = _plain(kind, x, gates, skip, state, lens, H, G, dim, vdim)
    # states and outputs of order one from some hundred 32-bit sums
    torch.testing.assert_close(out.double(), want, atol=2e-5, rtol=1e-4)
    torch.testing.assert_close(after.double(), want_state, atol=2e-5, rtol=1e-4)


@pytest.mark.parametrize("kind", ["delta", "selective"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_what_is_not_finite_reaches_no_earlier_token(kind, bad):
    H, G, dim, vdim, lens, at = 2, 1, 64, 20, [150], 120
    x, gates, skip, state = _inputs(kind, lens, H, G, dim, vdim, 3)
    clean, _ = _run(kind, x, gates, skip, state, lens, H, G, dim, vdim)
    x[at, 2 * G * dim + 5] = bad                                 # one value of head 0
    out, after = _run(kind, x, gates, skip, state, lens, H, G, dim, vdim)
    torch.testing.assert_close(out[:at], clean[:at], atol=1e-5, rtol=1e-5)
    others = torch.arange(H * vdim) != 5
    torch.testing.assert_close(out[:, others], clean[:, others], atol=1e-5, rtol=1e-5)
    assert not bool(torch.isfinite(out[at, 5])) and not bool(torch.isfinite(after[0, 5 * dim: 6 * dim]).any())
