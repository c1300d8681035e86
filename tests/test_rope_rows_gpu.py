"""Rotation and cache write of a step of many tokens from slabs of partial sums: the kernel of whole rows against the one of a wave per head (steps under 64 tokens),
which adds the same numbers in the same order and turns them by the same angles: equal to the bit."""
import pytest
import torch

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q, kv, hd, rot", [(3, 1, 8, 4), (40, 8, 128, 48), (64, 8, 128, 72), (7, 2, 40, 0)])
@pytest.mark.parametrize("parts", [1, 2, 3, 4, 6, 7])
@pytest.mark.parametrize("bias", [None, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cached", [True, False])
def test_rows_of_slabs(q, kv, hd, rot, parts, bias, cached):
    g = torch.Generator(device="cuda").manual_seed(q + parts)
    T, page = 100, 16
    heads = q + (2 if cached else 1) * kv
    slabs = torch.randn(parts, T, heads * hd, generator=g, device="cuda")
    b = torch.randn(heads * hd, generator=g, device="cuda").to(bias) if bias else None
    positions = torch.randint(0, 96, (T,), generator=g, device="cuda").int()
    req = torch.arange(T, device="cuda").int() // 7
    table = torch.randperm(15 * 6, generator=g, device="cuda").view(15, 6).int()          # (page 0 among them: its tokens are dropped)
    inv_freq = torch.rand(hd // 2, generator=g, device="cuda") if rot else None

    def run(cuts):
        qkv = torch.full((T, heads * hd), 7.0, dtype=torch.bfloat16, device="cuda")
        k, v = (torch.zeros(90, kv, page, hd, dtype=torch.bfloat16, device="cuda"), torch.zeros(90, kv, hd, page, dtype=torch.bfloat16, device="cuda")) if cached else (None, None)
        for a, e in cuts:
            planes = (req[a:e].contiguous(), table, k, v, page) if cached else ()
            ops.rope_cache_write(qkv[a:e], q, kv, hd, rot, positions[a:e].contiguous(), inv_freq, *planes, pairs=True, parts=slabs[:, a:e].contiguous(), bias=b)
        return [t for t in (qkv, k, v) if t is not None]

    # tokens that share a place would race: the later ones move to a free one
    seen = {}
    for t, (r, p) in enumerate(zip(req.tolist(), positions.tolist())):
        seen.setdefault((r, p), []).append(t)
    for same in list(seen.values()):
        for t in same[1:]:
            positions[t] = next(p for p in range(96) if (int(req[t]), p) not in seen)
            seen[(int(req[t]), int(positions[t]))] = [t]
    for x, y in zip(run([(0, T)]), run([(0, 63), (63, T)])):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))
