"""Which way latent attention takes for a step's long portions: sizes whose two ways differ by a fifth or more where both were measured."""
import pytest
import torch

from torchlet_amd.config.base import LatentAttentionSpec, PairRotarySpec
from torchlet_amd.engine.batch import StepContext
from torchlet_amd.parts.base import MIXERS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, rot, new, ctx, up", [
    (32, 64, [64], [8000], False), (16, 64, [64], [8000], False), (16, 64, [96], [16000], False), (8, 64, [64], [16000], False), (8, 64, [128], [8000], False),
    (16, 0, [64], [16000], False), (32, 64, [128], [8000], True), (16, 64, [256], [4000], True), (8, 64, [512], [8000], True), (16, 0, [96], [4000], True),
    (16, 64, [1024, 64], [0, 8000], True), (32, 64, [1] * 31 + [128], [2000] * 31 + [8000], True), (16, 64, [1] * 31 + [128], [2000] * 31 + [8000], True),
    (32, 64, [2048], [2048], True), (32, 64, [1] * 31 + [64], [2000] * 31 + [8000], True), (8, 64, [64], [40000], True)])
def test_the_faster_way(heads, rot, new, ctx, up):
    spec = LatentAttentionSpec(hidden=256, heads=heads, dim=128, rot_dim=rot, vdim=128, kv_rank=512, scale=0.07, norm_eps=1e-6, q_rank=0,
                               position=PairRotarySpec(dims=rot, base=1e4) if rot else None)
    part = MIXERS.build(spec, torch.bfloat16, "cuda")
    step = StepContext(new_lens=new, ctx_lens=ctx, slots=list(range(len(new))), token_ids=[0] * sum(new), want_rows=[], block_tables=[], tile_sizes=(), device="cuda")
    assert (part._portions(step, -(-step.max_total_len // 16)) is not None) == up
