"""The norm after a scaled sum with a row in registers: sizes on both sides of where its instances change, against the plain computation in 64 bits."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [4, 6, 1024, 1028, 2048, 2052, 4100, 8196, 16384, 16388])
@pytest.mark.parametrize("parts", [None, 0, 1, 2, 3, 4, 7, 9])
@pytest.mark.parametrize("dtype, with_out", [(torch.bfloat16, True), (torch.float32, True), (torch.float32, False)])
@pytest.mark.parametrize("weights", [torch.float32, torch.bfloat16])
def test_rows_in_registers(hidden, parts, dtype, with_out, weights):
    g = torch.Generator(device="cuda").manual_seed(hidden)
    rows = 3
    x = torch.randn(rows, hidden, generator=g, device="cuda")
    w = (1 + 0.1 * torch.randn(hidden, generator=g, device="cuda")).to(weights)
    pending = None if parts is None else torch.randn(rows, hidden, generator=g, device="cuda").to(dtype) if parts == 0 \
        else torch.randn(parts, rows, hidden, generator=g, device="cuda")
    r = 1.5 * x.double()
    if pending is not None:
        r = r + (pending.double() if parts == 0 else pending.double().sum(0))
    want = r / (r.pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * w.double()
    out = torch.empty(rows, hidden, dtype=dtype, device="cuda") if with_out else None
    ops.scaled_add_rmsnorm(x, pending, 1.5, w, 1e-5, out)
    # ten 32-bit additions of terms of up to four (1.5 x and the slabs, normal draws) round to 2^-24 of their partial sums each, which the norm divides by more
    # than one; the squares' sum and the root move a row by a few units of 2^-24 as a whole
    assert bool(((x.double() - want).abs() <= 2.0 ** -19 * (want.abs() + 1)).all())
    if with_out:
        assert torch.equal(out, x.to(dtype))


def test_rows_off_sixteen_bytes_keep_the_general_kernel():
    g = torch.Generator(device="cuda").manual_seed(1)
    x, y = torch.randn(2, 1024, generator=g, device="cuda"), torch.randn(2, 1024, generator=g, device="cuda").bfloat16()
    shifted = torch.empty(2 * 1024 + 1, dtype=torch.bfloat16, device="cuda")[1:].view(2, 1024)
    shifted.copy_(y)
    w = torch.ones(1024, device="cuda")
    a, b, oa, ob = x.clone(), x.clone(), torch.empty_like(y), torch.empty_like(y)
    ops.scaled_add_rmsnorm(a, y, 0.5, w, 1e-5, oa)
    ops.scaled_add_rmsnorm(b, shifted, 0.5, w, 1e-5, ob)
    assert bool(((a - b).abs() <= 2.0 ** -20 * (1 + a.abs())).all())
