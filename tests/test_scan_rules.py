"""The rules by which the recurrences choose a kernel for a step, called as the host calls them."""
import ctypes
from ctypes import c_int

import pytest

from torchlet_amd.kernels import build


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(str(build.build("recurrent", quiet=True)))


@pytest.mark.parametrize("lens, heads, dim, vdim, want", [
    ([2048], 16, 128, 128, 1), ([1] * 8 + [2048], 16, 128, 128, 1), ([1] * 31 + [512], 16, 128, 128, 1), ([512, 1, 1], 128, 128, 64, 1),      # decoded tokens beside one prompt
    ([700 - 75 * i for i in range(8)], 16, 128, 128, 1), ([512] * 16, 16, 128, 128, 2), ([1100, 825, 550, 275], 128, 128, 64, 2),
    ([1] * 64, 128, 128, 64, 1), ([4] * 64, 128, 128, 64, 1), ([512] * 16, 16, 256, 128, 1)])
def test_two_columns_a_lane_where_the_prompts_fill_the_gpu(lib, lens, heads, dim, vdim, want):
    assert lib.tl_delta_columns(*(c_int(x) for x in (dim, vdim, heads, len(lens), sum(lens), max(lens)))) == want


def _pays(lib, memory, lens, heads, dim, vdim):
    from torchlet_amd.kernels import ops
    p = ops.Portions.of(lens, 32)
    passes = -(-p.chunks * heads * (dim * vdim + dim + 1) // ops.CHUNK_SCRATCH)
    return bool(lib.tl_chunks_pay(*(c_int(x) for x in (memory, p.count, p.tokens, p.chunks, passes, p.longest, p.rest, p.rest_tokens, p.rest_longest, len(lens),
                                                       heads, dim, vdim))))


# steps whose two ways differ by a fifth or more where both were measured
@pytest.mark.parametrize("lens, heads, dim, vdim, want", [
    ([128], 16, 128, 128, False), ([512], 16, 128, 128, True), ([2048], 16, 128, 128, True), ([100] * 4, 16, 128, 128, False), ([33] * 40, 16, 128, 128, False),
    ([1] * 8 + [128], 16, 128, 128, False), ([1] * 31 + [64], 16, 128, 128, False), ([1] * 31 + [128], 16, 128, 128, False), ([1] * 31 + [512], 16, 128, 128, True),
    ([1] * 63 + [64], 16, 128, 128, False), ([1] * 63 + [512], 16, 128, 128, True), ([1] * 31 + [64] * 4, 16, 128, 128, False), ([1] * 31 + [2017], 16, 128, 128, True),
    ([1] * 8 + [64], 32, 128, 128, False), ([1] * 31 + [32], 32, 128, 128, False), ([20] * 8 + [128], 32, 128, 128, False), ([1] * 63 + [512], 32, 128, 128, True),
    ([128], 4, 64, 64, False), ([512], 4, 64, 64, True), ([1] * 63 + [128], 4, 64, 64, False), ([1] * 31 + [2017], 4, 64, 64, True)])
def test_fixed_decays_take_the_faster_way(lib, lens, heads, dim, vdim, want):
    assert _pays(lib, 0, lens, heads, dim, vdim) == want


@pytest.mark.parametrize("lens, heads, dim, vdim, want", [
    ([32], 4, 256, 512, False), ([64], 4, 256, 512, False), ([512], 4, 256, 512, True), ([100] * 4, 4, 256, 512, True), ([1] * 8 + [64], 4, 256, 512, True),
    ([1] * 31 + [64], 4, 256, 512, True), ([1] * 63 + [128], 4, 256, 512, True), ([1] * 31 + [2017], 8, 256, 512, True), ([20] * 8 + [32], 4, 256, 512, False),
    ([20] * 8 + [128], 4, 256, 512, True), ([1] * 200 + [256], 8, 256, 512, True), ([32], 2, 128, 128, False), ([1] * 31 + [64], 2, 128, 128, False),
    ([1] * 63 + [64], 2, 128, 128, True), ([1] * 31 + [64] * 4, 2, 128, 128, False), ([256], 2, 128, 128, True), ([1] * 200 + [256], 2, 128, 128, True)])
def test_the_matrix_memory_takes_the_faster_way(lib, lens, heads, dim, vdim, want):
    assert _pays(lib, 1, lens, heads, dim, vdim) == want


# the delta rule (1) and the selective recurrence (2): steps whose two ways differ by a tenth or more where both were measured
@pytest.mark.parametrize("mode, lens, heads, dim, vdim, want", [
    (1, [256], 16, 128, 128, True), (1, [2048], 16, 128, 128, True), (1, [175, 250, 325, 400], 16, 128, 128, True), (1, [1] * 15 + [256], 16, 128, 128, True),
    (1, [128] * 16, 32, 128, 128, False), (1, [275, 550, 825, 1100], 32, 128, 128, True), (1, [512], 4, 64, 64, True), (1, [128], 8, 256, 256, True),
    (2, [512], 128, 128, 64, True), (2, [275, 550, 825, 1100], 128, 128, 64, True), (2, [256], 64, 128, 64, True)])
def test_blocks_where_they_are_the_faster_way(lib, mode, lens, heads, dim, vdim, want):
    from torchlet_amd.kernels import ops
    p = ops.Portions.of(lens, ops.BLOCKS_FROM)
    assert bool(lib.tl_blocks_pay(*(c_int(x) for x in (mode, p.tokens, p.longest, p.rest, heads, dim, vdim)))) == want


# many portions whose work-groups outnumber the chip: the delta rule's loop is ahead, the selective recurrence's is not
@pytest.mark.parametrize("mode, lens, heads, dim, vdim, want", [
    (1, [128] * 64, 32, 128, 128, False), (1, [256] * 32, 32, 128, 128, False), (1, [128] * 64, 16, 128, 128, False), (1, [512] * 4, 32, 128, 128, True),
    (1, [128, 300, 500, 900], 32, 128, 128, True), (1, [512] * 4, 16, 128, 128, True), (2, [128] * 16, 128, 128, 64, True), (2, [256] * 32, 128, 128, 64, True)])
def test_blocks_of_crowded_steps(lib, mode, lens, heads, dim, vdim, want):
    from torchlet_amd.kernels import ops
    p = ops.Portions.of(lens, ops.BLOCKS_FROM)
    assert bool(lib.tl_blocks_pay(*(c_int(x) for x in (mode, p.tokens, p.longest, p.rest, heads, dim, vdim)))) == want
