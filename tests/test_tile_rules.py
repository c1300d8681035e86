"""The rules by which products choose a tile, called as the host calls them."""
import ctypes
from ctypes import c_int

import pytest

from torchlet_amd.kernels import build


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(str(build.build("gemm", quiet=True)))


# 1: 64 x 64, 2: 64 x 128, 3: 128 x 128; a launch has up to 65535 rows of tiles
@pytest.mark.parametrize("M, N, want", [(100, 3584, 1), (301, 37888, 2), (753, 37888, 3), (65535 * 64, 64, 1), (65535 * 64 + 1, 64, 3), (65535 * 64 + 1, 192, 3), (65535 * 128, 64, 3)])
def test_32_bit_tiles_fit_a_launch(lib, M, N, want):
    assert lib.tl_gemm_f32_tile(c_int(M), c_int(N)) == want
