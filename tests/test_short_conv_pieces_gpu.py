"""Short convolutions over whole pieces of four channels against the same numbers in rows that do not allow pieces (which the general kernels take), and against 64 bits."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _i32(x):
    return torch.tensor(x, dtype=torch.int32).cuda()


def _convolved(proj, conv, bias, tails, lens):
    """In 64 bits: silu of the convolution over each request's inputs behind its tail (``tails [requests, 3, C]``), and the tails behind them."""
    out, after, at = [], [], 0
    for r, n in enumerate(lens):
        rows = torch.cat((tails[r].double(), proj[at: at + n].double()))
        y = bias.double() + sum(rows[j: j + n] * conv.double()[:, j] for j in range(4))
        out.append(y / (1 + torch.exp(-y)))
        after.append(rows[n:])
        at += n
    return torch.cat(out), torch.stack(after)


# what a 32-bit convolution, silu and norm of numbers of order one make of 64 bits: a few roundings
CLOSE = dict(rtol=2e-6, atol=2e-6)


def _shift(t, by):
    """``t [T, C]`` as a view whose rows begin ``by`` numbers into rows ``by`` (mod 4, plus one) numbers longer."""
    wide = torch.zeros(t.shape[0], t.shape[1] + by + (1 if by else 0), dtype=t.dtype)
    wide[:, by: by + t.shape[1]] = t
    return wide.cuda()[:, by: by + t.shape[1]]


# one token each; as many tokens as requests, but two and none, or none to seven; portions in runs of two; portions in runs of eight that cross requests' ends
PLANS = [[1, 1, 1], [2, 0, 1, 1], [0, 0, 7, 0, 1, 3, 0, 0, 4, 0, 1, 2, 1, 1, 0, 2, 4, 0, 0, 0, 0, 4, 0, 0, 0, 0, 1, 0, 0, 0, 0], [5, 1, 3, 2], [700, 3, 1, 2, 1001, 8]]


@pytest.mark.parametrize("lens", PLANS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, kv, dim, vdim", [(16, 8, 128, 128), (6, 2, 4, 12), (40, 4, 256, 100)])
def test_delta(lens, dtype, heads, kv, dim, vdim):
    g = torch.Generator().manual_seed(3)
    T, R, C = sum(lens), len(lens), 2 * kv * dim + heads * vdim
    indptr = [0] + torch.tensor(lens).cumsum(0).tolist()
    req = _i32([r for r, n in enumerate(lens) for _ in range(n)])
    slots = _i32(list(range(R, 0, -1)))
    proj, conv = torch.randn(T, C, generator=g).to(dtype), torch.randn(C, 4, generator=g)
    gates, a_log, bias = torch.randn(T, 2 * heads, generator=g), torch.randn(heads, generator=g), torch.randn(heads, generator=g)
    start = torch.randn(R + 2, 8 + 3 * C, generator=g)
    got = []
    for by in (0, 1):
        state, gd, qkv = start.clone().cuda(), gates.clone().cuda(), torch.full((T, C), float("nan")).cuda()
        ops.delta_prepare(_shift(proj, by), conv.cuda(), gd, a_log.cuda(), bias.cuda(), state, 8, slots, _i32(indptr), req, qkv, heads, kv, dim, vdim, 4, 0.3, 1e-6)
        got.append((qkv.cpu(), gd.cpu(), state.cpu()))
    # queries and keys: the order of a head's sum of squares (up to 256 numbers: a few 32-bit roundings)
    torch.testing.assert_close(got[0][0], got[1][0], rtol=2e-6, atol=1e-7)
    assert torch.equal(got[0][0][:, 2 * kv * dim:], got[1][0][:, 2 * kv * dim:])
    assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][2], got[1][2])
    y, tails = _convolved(proj, conv, torch.zeros(C), start[slots.cpu().long(), 8:].view(R, 3, C), lens)
    unit = y[:, : 2 * kv * dim].view(T, 2 * kv, dim)
    unit = unit / torch.sqrt((unit * unit).sum(-1, keepdim=True) + 1e-6)
    unit[:, :kv] *= 0.3
    torch.testing.assert_close(got[0][0].double(), torch.cat((unit.flatten(1), y[:, 2 * kv * dim:]), 1), **CLOSE)
    z = gates.double()
    decay = torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(z[:, heads:] + bias.double()))
    torch.testing.assert_close(got[0][1].double(), torch.cat((torch.sigmoid(z[:, :heads]), decay), 1), **CLOSE)
    want = start.clone()
    want[slots.cpu().long(), 8:] = tails.float().reshape(R, -1)      # (inputs as they are: no rounding)
    assert torch.equal(got[0][2], want)


@pytest.mark.parametrize("lens", PLANS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, inner, gn", [(64, 4096, 128), (3, 12, 4)])
def test_selective(lens, dtype, heads, inner, gn):
    g = torch.Generator().manual_seed(4)
    T, R, C = sum(lens), len(lens), inner + 2 * gn
    indptr = [0] + torch.tensor(lens).cumsum(0).tolist()
    req = _i32([r for r, n in enumerate(lens) for _ in range(n)])
    slots = _i32(list(range(R, 0, -1)))
    proj, conv, conv_b = torch.randn(T, C + (heads + 3) // 4 * 4, generator=g).to(dtype), torch.randn(C, 4, generator=g), torch.randn(C, generator=g)
    a_log, bias = torch.randn(heads, generator=g), torch.randn(heads, generator=g)
    start = torch.randn(R + 2, 8 + 3 * C, generator=g)
    got = []
    for by in (0, 1):
        wide = torch.cat((torch.zeros(T, 4 + by, dtype=dtype), proj, torch.zeros(T, (4 - by) % 4, dtype=dtype)), 1).cuda()
        state, gd, out = start.clone().cuda(), torch.full((T, 2 * heads), float("nan")).cuda(), torch.full((T, C), float("nan")).cuda()
        ops.selective_prepare(wide, 4 + by, conv.cuda(), conv_b.cuda(), gd, a_log.cuda(), bias.cuda(), state, 8, slots, _i32(indptr), req, out, heads, inner, gn, 4)
        got.append((out.cpu(), gd.cpu(), state.cpu()))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    y, tails = _convolved(proj[:, :C], conv, conv_b, start[slots.cpu().long(), 8:].view(R, 3, C), lens)
    torch.testing.assert_close(got[0][0].double(), torch.cat((y[:, inner + gn:], y[:, inner: inner + gn], y[:, :inner]), 1), **CLOSE)
    dt = torch.nn.functional.softplus(proj[:, C: C + heads].double() + bias.double())
    torch.testing.assert_close(got[0][1].double(), torch.cat((dt, torch.exp(-torch.exp(a_log.double()) * dt)), 1), **CLOSE)
    want = start.clone()
    want[slots.cpu().long(), 8:] = tails.float().reshape(R, -1)
    assert torch.equal(got[0][2], want)


def test_one_request_beside_empty_ones_is_not_walked_token_by_token():
    heads, kv, dim, vdim, T = 16, 8, 128, 128, 2048
    C = 2 * kv * dim + heads * vdim
    g = torch.Generator().manual_seed(5)
    proj, conv, gates, a_log = (torch.randn(T, C, generator=g).bfloat16().cuda(), torch.randn(C, 4, generator=g).cuda(), torch.randn(T, 2 * heads, generator=g).cuda(),
                                torch.zeros(heads).cuda())
    indptr, req, slots = _i32([0] * 6 + [T] * (T - 5)), _i32([5] * T), _i32(list(range(T)))
    state, qkv = torch.zeros(T, 3 * C + 8).cuda(), torch.empty(T, C).cuda()

    def run():
        ops.delta_prepare(proj, conv, gates, a_log, a_log, state, 8, slots, indptr, req, qkv, heads, kv, dim, vdim, 4, 0.3, 1e-6)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    times = []
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        graph.replay()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) * 1e3)
    assert min(times) < 400                                  # (tens of us; 2048 tokens one after the other are more than a millisecond)
