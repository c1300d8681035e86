"""The choice between blocks of 16 tokens and the token loop as it is made: by a step's sizes, and what it does to a portion's numbers."""
from ctypes import c_int

import pytest
import torch
from test_recurrence_blocks_gpu import _inputs, _plain, _run

from torchlet_amd.kernels import ops

pytestmark = pytest.mark.gpu

# What a 32-bit result may differ by: outputs and states are sums of some hundred products of numbers up to a few units, each rounded at 2^-24 of its size; relative to the whole
# tensor (2-norms) a few of them.
FEW_ROUNDINGS = 4 * 2.0 ** -24


def _error(got, want):
    return float((got.double() - want).norm() / want.norm())


def _pays(kind, lens, H, dim, vdim):
    p = ops.Portions.of(lens, ops.BLOCKS_FROM)
    return bool(p.count and ops._lib("recurrent").tl_blocks_pay(*(c_int(x) for x in (1 if kind == "delta" else 2, p.tokens, p.longest, p.rest, H, dim, vdim))))


def _step(kind, lens, H, G, dim, vdim, rows):
    x, gates, skip, state = rows
    T = sum(lens)
    return _run(kind, x[:T].contiguous(), gates[:T].contiguous(), skip, state[: len(lens)].contiguous(), lens, H, G, dim, vdim, portions=ops.Portions.of(lens, ops.BLOCKS_FROM))


# a portion alone and beside others: beside the first company the rule takes the other way for it, beside the second the same
@pytest.mark.parametrize("kind, H, G, dim, vdim, own, flips, keeps", [
    ("delta", 16, 8, 128, 128, 128, [1] * 31, [300]), ("delta", 32, 16, 128, 128, 128, [128] * 15, [600, 200]), ("selective", 128, 1, 128, 64, 128, [1] * 31, [300])])
def test_a_portion_alone_and_in_company(kind, H, G, dim, vdim, own, flips, keeps):
    assert _pays(kind, [own], H, dim, vdim) and not _pays(kind, [own] + flips, H, dim, vdim) and _pays(kind, [own] + keeps, H, dim, vdim)
    rows = _inputs(kind, [own] + [max(sum(flips), sum(keeps))] + [0] * max(len(flips), len(keeps)), H, G, dim, vdim, 11)
    alone, alone_state = _step(kind, [own], H, G, dim, vdim, rows)
    same, same_state = _step(kind, [own] + keeps, H, G, dim, vdim, rows)
    other, other_state = _step(kind, [own] + flips, H, G, dim, vdim, rows)
    assert torch.equal(same[:own], alone) and torch.equal(same_state[0], alone_state[0])
    assert not torch.equal(other[:own], alone)
    x, gates, skip, state = rows
    want, want_state = _plain(kind, x[:own], gates[:own], skip, state[:1], [own], H, G, dim, vdim)
    for out, after in ((alone, alone_state), (other[:own], other_state)):
        assert _error(out, want) < FEW_ROUNDINGS and _error(after[0], want_state[0]) < FEW_ROUNDINGS


# below the blocks' least the loop has every portion, whatever is beside it
@pytest.mark.parametrize("kind", ["delta", "selective"])
def test_short_portions_keep_their_bits(kind):
    H, G, dim, vdim, own = 8, 4, 64, 32, ops.BLOCKS_FROM - 1
    rows = _inputs(kind, [own, 600, 0], H, G, dim, vdim, 12)
    alone, alone_state = _step(kind, [own], H, G, dim, vdim, rows)
    beside, beside_state = _step(kind, [own, 500, 2], H, G, dim, vdim, rows)
    assert torch.equal(beside[:own], alone) and torch.equal(beside_state[0], alone_state[0])


# a step whose blocks' matrices would be more than the scratch holds is the loop's, to the bit
@pytest.mark.parametrize("kind", ["delta", "selective"])
def test_more_than_the_scratch_holds(kind, monkeypatch):
    H, G, dim, vdim, lens = 8, 4, 64, 32, [400, 1, 200]
    assert _pays(kind, lens, H, dim, vdim)
    rows = _inputs(kind, lens, H, G, dim, vdim, 13)
    x, gates, skip, state = rows
    blocks, _ = _step(kind, lens, H, G, dim, vdim, rows)
    loop, loop_state = _run(kind, x, gates, skip, state, lens, H, G, dim, vdim, portions=ops.Portions.of(lens, 1 << 30))
    p = ops.Portions.of(lens, ops.BLOCKS_FROM)
    floats = ops._lib("recurrent").tl_blocks_floats(c_int(1 if kind == "delta" else 2), c_int(p.tokens // 16 + p.count), c_int(H))
    monkeypatch.setattr(ops, "CHUNK_SCRATCH", floats - 1)
    out, after = _step(kind, lens, H, G, dim, vdim, rows)
    assert torch.equal(out, loop) and torch.equal(after, loop_state) and not torch.equal(out, blocks)


# whole outputs of long portions against 64 bits: as close in blocks as in the loop
@pytest.mark.parametrize("kind, H, G, dim, vdim", [("delta", 16, 8, 128, 128), ("delta", 4, 4, 64, 64), ("selective", 32, 1, 128, 64)])
def test_errors_of_long_portions(kind, H, G, dim, vdim):
    lens = [700]
    assert _pays(kind, lens, H, dim, vdim)
    rows = _inputs(kind, lens, H, G, dim, vdim, 14)
    x, gates, skip, state = rows
    want, want_state = _plain(kind, x, gates, skip, state, lens, H, G, dim, vdim)
    blocks = _step(kind, lens, H, G, dim, vdim, rows)
    loop = _run(kind, x, gates, skip, state, lens, H, G, dim, vdim, portions=ops.Portions.of(lens, 1 << 30))
    for got, of_loop, to in zip(blocks, loop, (want, want_state)):
        print(kind, H, dim, "blocks", _error(got, to), "loop", _error(of_loop, to))
        assert _error(got, to) < min(FEW_ROUNDINGS, 1.25 * _error(of_loop, to))
