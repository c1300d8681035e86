"""Latent attention over long portions of prompts: keys and values projected up for the step, against the absorbed way over the cached rows.

The two differ in what is rounded to bfloat16 between the products (the projected query, the weights and the mixed latent, or keys, values and the weights): at most
eight independent roundings of 2^-9 each on the way to an output, 2^-7.5 of its size; held here to 2^-6 of a token's norm."""
from types import SimpleNamespace

import pytest
import torch

from torchlet_amd.config.base import HalfRotarySpec, LatentAttentionSpec, PairRotarySpec
from torchlet_amd.engine.batch import StepContext
from torchlet_amd.kernels import ops
from torchlet_amd.parts import latent_attention
from torchlet_amd.parts.base import MIXERS

pytestmark = pytest.mark.gpu


def _mixer(heads, dim, rot, vdim, rank, g, halves=False, **more):
    spec = LatentAttentionSpec(hidden=256, heads=heads, dim=dim, rot_dim=rot, vdim=vdim, kv_rank=rank, scale=(dim + rot) ** -0.5, norm_eps=1e-6,
                               position=(HalfRotarySpec if halves else PairRotarySpec)(dims=rot, base=10000.0) if rot else None, **more)
    part = MIXERS.build(spec, torch.bfloat16, "cuda")
    part.load_weights({k: torch.randn(*w.shape, generator=g) * w.shape[-1] ** -0.5 if len(w.shape) > 1 else 1 + 0.1 * torch.randn(*w.shape, generator=g)
                       for k, w in part.weight_specs().items()})
    return part


def _ctx(new, ctx, page, tables):
    return StepContext(new_lens=new, ctx_lens=ctx, slots=list(range(len(new))), token_ids=[0] * sum(new), want_rows=[], block_tables=[tables], tile_sizes=(),
                       device="cuda")


@pytest.mark.parametrize("form", [dict(q_rank=192, sink=True), dict(q_rank=0, gate_values=True), dict(q_rank=0, window=100, gate_values=True),
                                  dict(q_rank=64, window=64, gate=True, sink=True)])
@pytest.mark.parametrize("heads, dim, rot, vdim, rank", [(4, 128, 64, 128, 512), (20, 128, 0, 128, 64), (3, 64, 0, 64, 128)])
@pytest.mark.parametrize("page, halves", [(16, False), (24, True)])
def test_long_portions_project_keys_and_values_up(form, heads, dim, rot, vdim, rank, page, halves, monkeypatch):
    monkeypatch.setattr(latent_attention, "_UP_LEAST", 0)          # (steps of this size stay with the absorbed way otherwise)
    monkeypatch.setattr(latent_attention, "_UP_LEAST_BESIDE", 0)
    g = torch.Generator().manual_seed(heads + page)
    part = _mixer(heads, dim, rot, vdim, rank, g, halves, **form)
    assert part.project_up
    new, ctx = [1, 128, 63, 333, 64, 129], [200, 0, 31, 257, 0, 63]
    blocks = [-(-(n + c) // page) for n, c in zip(new, ctx)]
    tables = torch.zeros(len(new), max(blocks), dtype=torch.int32)
    order = 1 + torch.randperm(sum(blocks), generator=g)
    at = 0
    for r, b in enumerate(blocks):
        first = max(0, ctx[r] - part.window + 1) // page if part.window else 0      # (pages wholly before the window are given back)
        tables[r, first:b] = order[at + first: at + b].int()
        at += b
    cached = (torch.randn(1 + sum(blocks), 1, page, rank + rot, generator=g)).bfloat16().cuda()
    cached[0] = float("nan")
    h = torch.randn(sum(new), 256, generator=g).bfloat16().cuda()

    def run(up, step, rows, scratch=None):
        monkeypatch.setattr(part, "project_up", up)
        if scratch:
            monkeypatch.setattr(ops, "PROMPT_ROWS_SCRATCH_BYTES", scratch)
        plane = cached.clone()
        out = part.forward(rows, step, SimpleNamespace(planes=(plane,), group=0, page_size=page, writable=True))
        return (out.float().sum(0) if out.dim() == 3 else out.float()), plane

    def same(a, b):
        assert bool(torch.isfinite(b[0]).all()) and torch.equal(a[1].nan_to_num(), b[1].nan_to_num())
        assert bool(((a[0] - b[0]).norm(dim=1) <= 2.0 ** -6 * b[0].norm(dim=1)).all()), float(((a[0] - b[0]).norm(dim=1) / b[0].norm(dim=1)).max())

    step = _ctx(new, ctx, page, tables.numpy())
    want = run(False, step, h)
    same(run(True, step, h), want)                         # beside a decoded token and short portions
    held = step.long_portions(64, part.window)[4] * (dim + vdim) * 2
    same(run(True, step, h, scratch=held * 2), want)       # two heads' keys and values at once (and one, where the heads are odd)
    same(run(True, step, h, scratch=held - 1), want)       # not even one head's: the absorbed way
    alone = _ctx([333], [257], page, tables[3:4].numpy())
    same(run(True, alone, h[192: 192 + 333], scratch=1 << 30), run(False, alone, h[192: 192 + 333]))
