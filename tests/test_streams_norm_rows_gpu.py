"""The norm over several copies of the residual at every kind of width and number of copies its kernels part at."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 3, 4])
@pytest.mark.parametrize("width", [4, 1028, 4096, 4100, 8196, 70])
def test_norm_over_copies_at_every_width_of_its_kernels(S, width):
    """Rows in registers (widths of whole pieces, 1, 2 or 4 copies) and the general kernel against 64 bits, with and without pending output."""
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(width + S)
    T, eps = 5, 1e-5
    x = torch.randn(S, T, width, generator=g)
    mix, gate, read = torch.eye(S) + 0.1 * torch.randn(S, S, generator=g), torch.randn(S, generator=g), torch.randn(S, generator=g)
    w, b = torch.randn(width, generator=g), torch.randn(width, generator=g)
    for pending in (None, torch.randn(T, width, generator=g).bfloat16(), torch.randn(3, T, width, generator=g)):
        dev = x.clone().cuda()
        out = torch.empty(T, width, dtype=torch.bfloat16, device="cuda")
        ops.streams_norm(dev, None if pending is None else pending.cuda(), None if pending is None else (mix.cuda(), gate.cuda()), read.cuda(), "layernorm",
                         w.cuda(), b.cuda(), eps, out)
        xs = x.double()
        if pending is not None:
            p = pending.double() if pending.dim() == 2 else pending.double().sum(0)
            xs = torch.stack([sum(mix[a, c].double() * xs[a] for a in range(S)) + gate[c].double() * p for c in range(S)])
        u = sum(read[a].double() * xs[a] for a in range(S))
        d = u - u.mean(-1, keepdim=True)
        want = d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w.double() + b.double()
        torch.testing.assert_close(dev.cpu().double(), xs, rtol=1e-6, atol=1e-5)
        torch.testing.assert_close(out.cpu().double(), want, rtol=2.0 ** -8, atol=1e-4)


@pytest.mark.parametrize("S", [1, 2, 3, 4])
@pytest.mark.parametrize("width", [1028, 4100, 70])
@pytest.mark.parametrize("kind, gain", [("layernorm", 0.7), ("rmsnorm", 1.3)])
def test_chosen_rows_kinds_and_float_output(S, width, kind, gain):
    """Chosen rows take the pending output in without leaving it in the copies; both kinds of norm with a gain; 32-bit outputs."""
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(width + S)
    T, eps, rows = 7, 1e-5, [6, 0, 3]
    x = torch.randn(S, T, width, generator=g)
    mix, gate, read = torch.eye(S) + 0.1 * torch.randn(S, S, generator=g), torch.randn(S, generator=g), torch.randn(S, generator=g)
    w, b = torch.randn(width, generator=g), torch.randn(width, generator=g)
    for pending in (None, torch.randn(T, width, generator=g), torch.randn(2, T, width, generator=g)):
        dev = x.clone().cuda()
        out = torch.empty(len(rows), width, dtype=torch.float32, device="cuda")
        ops.streams_norm(dev, None if pending is None else pending.cuda(), None if pending is None else (mix.cuda(), gate.cuda()), read.cuda(), kind,
                         w.cuda(), b.cuda() if kind == "layernorm" else None, eps, out, rows=torch.tensor(rows, dtype=torch.int32, device="cuda"), gain=gain)
        assert torch.equal(dev.cpu(), x)
        xs = x.double()
        if pending is not None:
            p = pending.double() if pending.dim() == 2 else pending.double().sum(0)
            xs = torch.stack([sum(mix[a, c].double() * xs[a] for a in range(S)) + gate[c].double() * p for c in range(S)])
        u = sum(read[a].double() * xs[a] for a in range(S))[rows]
        if kind == "layernorm":
            d = u - u.mean(-1, keepdim=True)
            want = (d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w.double() + b.double()) * gain
        else:
            want = u / torch.sqrt((u * u).mean(-1, keepdim=True) + eps) * gain * w.double()
        # (32-bit sums of some ten terms, a mean over the row and a handful of products: a few units of 2^-24 each)
        torch.testing.assert_close(out.cpu().double(), want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("S,width,rows", [(1, 2048, 3), (4, 2048, 300), (1, 8196, 256), (2, 8192, 257), (4, 8192, 300), (1, 15360, 300), (2, 15360, 3)])
@pytest.mark.parametrize("kind", ["layernorm", "rmsnorm"])
@pytest.mark.parametrize("slabs", [0, 3, 9])
def test_vectors_at_any_address_and_any_number_of_rows_give_the_same_bits(S, width, rows, kind, slabs):
    """The norm's vectors behind one more number (no whole pieces to fetch them in), and rows beyond those that have a compute unit each: the registers' kernel all the same, number by number
    and later instead of in whole pieces and at once, with the same sums."""
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(width + rows)
    x, pending = torch.randn(S, rows, width, generator=g), torch.randn(*((slabs,) if slabs else ()), rows, width, generator=g)
    pending = (pending if slabs else pending.bfloat16()).cuda()
    vectors = [torch.randn(width + 8, generator=g).to(torch.bfloat16 if kind == "layernorm" else torch.float32).cuda() for _ in range(2)]

    def norm(n, at):
        w, b = (torch.cat((v[:at], v)).cuda()[at: at + width] for v in vectors)
        copies, out = x[:, :n].contiguous().cuda(), torch.empty(n, width, dtype=torch.bfloat16, device="cuda")
        ops.streams_norm(copies, (pending[:, :n] if slabs else pending[:n]).contiguous(), None, None, kind, w, b if kind == "layernorm" else None, 1e-5, out)
        return copies, out

    copies, want = norm(rows, 0)
    for n, at in ((rows, 1), (rows, 4), (2, 0), (2, 3)):
        got = norm(n, at)
        assert torch.equal(got[1], want[:n]) and torch.equal(got[0], copies[:, :n])
