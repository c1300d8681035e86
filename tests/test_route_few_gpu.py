"""The router's choice up to 16 tokens and up to 64 experts (one launch, an expert to a lane) against the general walk, which more experts take: the same choices, weights and sort
around both limits, with ties, infinities and outputs that are no numbers."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 5, 16, 17])
@pytest.mark.parametrize("experts,top,scores,groups", [(1, 1, "all", None), (16, 2, "chosen", None), (18, 3, "all", None), (64, 8, "sigmoid", (8, 3)), (24, 24, "chosen", None), (20, 2, "all", (4, 2))])
def test_choice_by_lanes_is_the_choice_of_the_walk(tokens, experts, top, scores, groups):
    from torchlet_amd.kernels import ops
    g = torch.Generator().manual_seed(tokens * 100 + experts)
    z = torch.randn(tokens, experts, generator=g).mul(4).round().div(2)          # ties among them
    if tokens > 1 and experts > top:
        z[1, 0], z[1, 1] = float("nan"), float("-inf")
        z[0, experts - 1] = float("-inf")
    bias = torch.randn(experts, generator=g) * 0.25 if scores != "chosen" else None
    weights, offsets, slot_token, pair_slot = ops.route(z.cuda(), top, scores, None if bias is None else bias.cuda(), 1.5, 1e-20, groups)
    # beside groups of experts that lose against every other one the walk has more than 64 to go through
    size = experts if groups is None else experts // groups[0]
    more = -(-65 // size) * size
    wide = torch.cat((z, torch.full((tokens, more), float("-inf"))), 1)
    wide_bias = None if bias is None else torch.cat((bias, torch.full((more,), -1e30)))
    ref = ops.route(wide.cuda(), top, scores, None if wide_bias is None else wide_bias.cuda(), 1.5, 1e-20, None if groups is None else (groups[0] + more // size, groups[1]))
    sane = [t for t in range(tokens) if not z[t].isnan().any()]
    assert torch.equal(weights.cpu()[sane], ref[0].cpu()[sane])
    chosen = torch.empty(tokens * top, dtype=torch.long)
    chosen_ref = torch.empty_like(chosen)
    for out, off, pairs, n in ((chosen, offsets, pair_slot, experts), (chosen_ref, ref[1], ref[3], experts + more)):
        slots = torch.repeat_interleave(torch.arange(n), torch.diff(off.cpu().long()))
        out.copy_(slots[pairs.cpu().long()])
    for t in sane:
        assert torch.equal(chosen[t * top: (t + 1) * top], chosen_ref[t * top: (t + 1) * top])
    assert sorted(pair_slot.tolist()) == list(range(tokens * top))
    assert [slot_token.tolist()[s] for s in pair_slot.tolist()] == [i // top for i in range(tokens * top)]
    if tokens > 1 and experts > top:                 # what is no number is not chosen while a number is left
        picked = chosen[top: 2 * top].tolist()
        assert scores == "all" or 0 not in picked
