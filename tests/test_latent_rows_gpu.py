"""Some tokens' queries and gates brought side by side and their rows put back, against indexing."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, dim, rot, rank, extra, gate_cols", [(4, 128, 64, 512, 16, 4), (20, 128, 0, 64, 8, 20 * 128), (3, 64, 8, 128, 0, 0), (16, 128, 64, 512, 8, 16)])
@pytest.mark.parametrize("tokens", [[0], [6, 2, 3], list(range(0, 7))])
def test_rows_taken_and_put_back(heads, dim, rot, rank, extra, gate_cols, tokens):
    g = torch.Generator().manual_seed(heads + len(tokens))
    T, n, at = 7, len(tokens), heads * (dim + rot)
    down = torch.randn(T, at + extra + gate_cols + (-(at + extra + gate_cols)) % 8, generator=g).bfloat16().cuda()
    q, gate = down[:, :at], down[:, at + extra: at + extra + gate_cols] if gate_cols else None
    idx = torch.tensor(tokens, dtype=torch.int32, device="cuda")
    own = torch.empty(n, heads * dim, dtype=torch.bfloat16, device="cuda")
    qrow = torch.zeros(n, heads * (rank + rot), dtype=torch.bfloat16, device="cuda")
    gates = torch.empty(n, gate_cols, dtype=torch.bfloat16, device="cuda") if gate_cols else None
    ops.latent_take(q, heads, dim, rot, idx, own, qrow, rank, gate, gates)
    want = q[idx.long()].view(n, heads, dim + rot)
    assert torch.equal(own.view(n, heads, dim), want[:, :, :dim]) and torch.equal(qrow.view(n, heads, rank + rot)[:, :, rank:], want[:, :, dim:])
    assert not bool(qrow.view(n, heads, rank + rot)[:, :, :rank].any())
    if gate_cols:
        assert torch.equal(gates, gate[idx.long()])
    dst = torch.zeros(T, heads * dim + 8, dtype=torch.bfloat16, device="cuda")
    ops.put_rows(own, idx, dst[:, : heads * dim])
    back = torch.zeros_like(dst)
    back[idx.long(), : heads * dim] = own
    assert torch.equal(dst, back)
