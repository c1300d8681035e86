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
