"""Rows held in registers: the gated norm over stretches of every size class, embedding rows and the sum of two normed branches."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _tol(dtype):
    # one rounding of the result (2^-9 of its size for bfloat16), or a few 32-bit roundings
    return dict(rtol=2 ** -8, atol=1e-6) if dtype == torch.bfloat16 else dict(rtol=2e-5, atol=1e-6)


# last of a class, first of the next, a stretch with idle lanes, one that is no multiple of four and one beyond the largest class
@pytest.mark.parametrize("vdim", [4, 64, 68, 128, 132, 256, 260, 512, 516, 2048, 2052, 4096, 4100, 8192, 8196, 16384, 16388, 510, 1026])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("stored", [torch.float32, torch.bfloat16])
def test_gated_norm(vdim, dtype, stored):
    g = torch.Generator().manual_seed(vdim)
    T, H = 5, 1 if vdim > 512 else 3
    o = torch.randn(T, H * vdim, generator=g)
    gate = torch.randn(T, H * vdim + 8, generator=g).to(dtype)
    w = torch.randn(H * vdim, generator=g).to(stored)
    for first, kind in ((False, "sigmoid"), (True, "silu")):
        out = torch.full((T, H * vdim), 7.0, dtype=dtype).cuda()
        ops.gated_head_norm(o.cuda(), gate.cuda()[:, 8:], w.cuda(), 1e-5, out, H, vdim, gate=kind, gain=0.7, gate_first=first)
        z = gate[:, 8:].double()
        f = (torch.sigmoid(z) * (z if kind == "silu" else 1.0)).view(T, H, vdim)
        x = o.double().view(T, H, vdim)
        s = x * f if first else x
        want = x * f / torch.sqrt((s * s).mean(-1, keepdim=True) + 1e-5) * w.double().view(1, H, vdim) * 0.7
        torch.testing.assert_close(out.cpu().double().view(T, H, vdim), want, **_tol(dtype))


@pytest.mark.parametrize("hidden", [4, 256, 260, 4096, 4100, 8196, 12288, 510])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embedding_and_branches(hidden, dtype):
    g = torch.Generator().manual_seed(hidden)
    V, T = 11, 6
    table, big = torch.randn(V, hidden, generator=g).to(dtype), torch.randn(8, hidden, generator=g).to(dtype)
    ids = torch.tensor([3, 10, 0, 3, 7, 1], dtype=torch.int32)
    pos_table = torch.randn(9, hidden, generator=g)
    pos = torch.tensor([0, 1, 2, 8, 0, 5], dtype=torch.int32)
    for copies in (1, 3):
        out = torch.empty((copies, T, hidden) if copies > 1 else (T, hidden)).cuda()
        ops.embedding(ids.cuda(), table.cuda(), out, 0.5, pos.cuda(), pos_table.cuda())
        want = table.float()[ids.long()] * 0.5 + pos_table[pos.long()]
        assert torch.equal(out.cpu(), want.expand(out.shape))
    w = torch.randn(hidden, generator=g)
    out = torch.empty(T, hidden).cuda()
    ops.embedding_norm(ids.cuda(), table.cuda(), out, 2.0, w.cuda(), 1e-5)
    x = table.double()[ids.long()] * 2.0
    torch.testing.assert_close(out.cpu().double(), x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.double(), rtol=2e-5, atol=1e-6)
    # bigram rows: as many tokens as requests (one of them with none, one with two), and more tokens than requests
    for indptr, positions in (([0, 1, 3, 3, 4, 5, 6], [4, 0, 1, 0, 7, 2]), ([0, 4, 6], [3, 4, 5, 6, 0, 1])):
        R = len(indptr) - 1
        req = torch.repeat_interleave(torch.arange(R), torch.tensor(indptr).diff()).to(torch.int32)
        slots = torch.arange(R, dtype=torch.int32).flip(0).contiguous()
        last = torch.arange(R, dtype=torch.int32).view(R, 1) + 1
        kept = last.clone()
        out, dev_last = torch.empty(T, hidden).cuda(), last.cuda()
        ops.bigram_embedding(ids.cuda(), table.cuda(), out, 0.5, big.cuda(), 7, 5, 3, req.cuda(), torch.tensor(indptr, dtype=torch.int32).cuda(),
                             torch.tensor(positions, dtype=torch.int32).cuda(), slots.cuda(), dev_last)
        for t in range(T):
            r = int(req[t])
            before = int(ids[t - 1]) if t > indptr[r] else int(kept[int(slots[r])])
            row = 7 if positions[t] == 0 else (before * 5 + int(ids[t]) * 3) % 7
            torch.testing.assert_close(out[t].cpu().double(), table.double()[int(ids[t])] * 0.5 + big.double()[row], rtol=1e-6, atol=1e-6)
        for r in range(R):
            want = int(ids[indptr[r + 1] - 1]) if indptr[r + 1] > indptr[r] else int(kept[int(slots[r])])
            assert int(dev_last[int(slots[r])]) == want
    for B in (2, 3):
        x, w = torch.randn(B, T, hidden, generator=g).to(dtype), torch.randn(B, hidden, generator=g)
        out = torch.empty(T, hidden, dtype=dtype).cuda()
        ops.normed_sum(x.cuda(), w.cuda(), 1e-5, out)
        want = (x.double() / torch.sqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()[:, None]).sum(0)
        torch.testing.assert_close(out.cpu().double(), want, rtol=2 ** -8 if dtype == torch.bfloat16 else 2e-5, atol=1e-5)


def _graph_us(fn):
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    times = []
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        graph.replay()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) * 1e3)
    return min(times)


def test_bigram_rows_of_one_request_beside_empty_ones():
    """As many tokens as requests, all of them one request's: the rows, the token that is kept, and a time that no walk from token to token fits in."""
    T, hidden, V, ids = 2048, 256, 50, torch.randint(0, 50, (2048,), generator=torch.Generator().manual_seed(1), dtype=torch.int32)
    g = torch.Generator().manual_seed(2)
    table, big = torch.randn(V, hidden, generator=g), torch.randn(8, hidden, generator=g)
    at = 1000                                                # the request's number; those before it end at token 0, those behind it at T
    indptr = torch.tensor([0] * (at + 1) + [T] * (T - at), dtype=torch.int32)
    req = torch.full((T,), at, dtype=torch.int32)
    positions, slots = torch.arange(3, 3 + T, dtype=torch.int32), torch.arange(T, dtype=torch.int32)
    last = torch.full((T, 1), 9, dtype=torch.int32).cuda()
    out = torch.empty(T, hidden).cuda()
    args = [t.cuda() for t in (big, req, indptr, positions, slots, ids, table)]
    big_d, req_d, indptr_d, positions_d, slots_d, ids_d, table_d = args

    def run():
        ops.bigram_embedding(ids_d, table_d, out, 0.5, big_d, 7, 5, 3, req_d, indptr_d, positions_d, slots_d, last)
    run()
    before = torch.cat((torch.tensor([9]), ids[:-1].long()))
    want = table.double()[ids.long()] * 0.5 + big.double()[(before * 5 + ids.long() * 3) % 7]
    torch.testing.assert_close(out.cpu().double(), want, rtol=1e-6, atol=1e-6)
    kept = torch.full((T,), 9, dtype=torch.int32)
    kept[at] = ids[-1]
    assert torch.equal(last.cpu()[:, 0], kept)
    assert _graph_us(run) < 300                              # (tens of us; 2048 rows one after the other are a millisecond)
