"""The recurrences where a step has more requests and heads than the GPU holds work-groups of one column a lane: two columns to a lane, the same
bits as every request alone, outputs and states."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["delta", "decay", "selective"])
@pytest.mark.parametrize("dim, vdim", [(64, 40), (128, 36), (100, 33), (36, 50)])
def test_many_requests_give_the_bits_of_each_alone(kind, dim, vdim):
    from torchlet_amd.kernels import ops
    H, R = 8, 64                                   # 3 or 4 tiles of 16 columns x 8 heads x 64 requests: more than 1024
    G = H if kind == "decay" else 2
    gen = torch.Generator(device="cuda").manual_seed(dim)
    lens = [5 + (i * 11) % 27 for i in range(R)]
    T, C = sum(lens), 2 * G * dim + H * vdim
    x = torch.randn(T, C, generator=gen, device="cuda") * 0.3
    gates = torch.rand(T, 2 * H, generator=gen, device="cuda") * 0.9 + 0.05
    head = torch.rand(H, generator=gen, device="cuda")
    start = torch.randn(R, H * dim * vdim, generator=gen, device="cuda")

    def run(x, gates, state, lens):
        out = torch.full((x.shape[0], H * vdim), float("nan"), device="cuda")
        slots = torch.arange(len(lens), dtype=torch.int32, device="cuda")
        indptr = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
        most = max(max(lens), 16)                  # (batches of 16 tokens in every call)
        if kind == "delta":
            ops.delta_scan(x, gates, state, slots, indptr, out, H, G, dim, vdim, max_new_tokens=most)
        elif kind == "decay":
            ops.decay_scan(x, head, state, slots, indptr, out, H, dim, vdim, max_new_tokens=most)
        else:
            ops.selective_scan(x, gates, head, state, slots, indptr, out, H, G, dim, vdim, max_new_tokens=most)
        return out

    state = start.clone()
    out = run(x, gates, state, lens)
    assert bool(torch.isfinite(out).all())
    at = 0
    for r, n in enumerate(lens):
        alone = start[r: r + 1].clone()
        got = run(x[at: at + n].contiguous(), gates[at: at + n].contiguous(), alone, [n])
        assert torch.equal(got, out[at: at + n]) and torch.equal(alone[0], state[r]), r
        at += n
