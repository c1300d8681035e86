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
