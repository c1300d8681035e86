"""How a step's long portions are cut into passes over the chunks' scratch: by the portions alone, within the bound on the scratch."""
import pytest

from torchlet_amd.kernels import ops


class _Pays:
    @staticmethod
    def tl_chunks_pay(*_):
        return 1


def _plan(lens, heads=8, dim=256, vdim=512, exact=True):
    portions = ops.Portions.of(lens, ops.CHUNKED_FROM) if exact else ops.Portions.bound(sum(lens), len(lens), None, ops.CHUNKED_FROM)
    return ops._chunk_scratch(_Pays, True, len(lens), heads, dim, vdim, 0, "meta", portions)


@pytest.mark.parametrize("decoded", [0, 30, 31, 255])
def test_decoded_requests_take_no_part_of_the_scratch(decoded):
    # 63 chunks of 8 heads of 256 x 512 fit: a portion of 2017 tokens is 32
    plan = _plan([1] * decoded + [2017])
    assert plan.segment >= 2017 and plan.grid == 32 and plan.scratch.numel() == plan.floats <= ops.CHUNK_SCRATCH


@pytest.mark.parametrize("lens, passes", [([1024] * 8, 3), ([2048], 1), ([64 * 63], 1), ([64 * 63 + 1], 2), ([40] * 63, 1), ([6000, 40], 4)])
def test_passes_are_as_many_as_the_scratch_asks_for(lens, passes):
    plan = _plan(lens)
    assert -(-max(lens) // plan.segment) == passes
    per_chunk = 8 * (256 * 512 + 256 + 1)
    assert plan.grid * per_chunk <= plan.floats <= ops.CHUNK_SCRATCH
    # no pass holds more chunks than the grid has
    for at in range(0, max(lens), plan.segment):
        assert sum(-(-min(max(n - at, 0), plan.segment) // 64) for n in lens) <= plan.grid


@pytest.mark.parametrize("lens", [[40] * 64, [4] * 64, [1] * 300, [31]])
def test_portions_that_do_not_fit_or_are_none_leave_it_to_the_token_loop(lens):
    assert _plan(lens) is None


@pytest.mark.parametrize("lens", [[65, 0], [0, 300, 1], [32] * 5, [31] * 9, [1, 200, 64], [20]])
def test_bounds_hold_what_there_is(lens):
    exact, bound = ops.Portions.of(lens, 32), ops.Portions.bound(sum(lens), len(lens), None, 32)
    assert all(b >= e for b, e in zip(bound[:4], exact[:4])) or bound.count == 0
    assert bound.rest >= exact.rest and bound.rest_longest >= min(exact.rest_longest, 31)
