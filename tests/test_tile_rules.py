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


# one row of tiles against wide matrices, measured 10 % and more apart: not 64 x 64 with more work-groups than compute units unless the rows of w lie multiples of 4 KB apart or are short, and with the
# fused gate not four slabs of few work-groups
@pytest.mark.parametrize("M, N, K, gated, ahead", [
    (63, 18944, 5120, 0, [(64, 128), (128, 128)]), (63, 18944, 3584, 0, [(64, 128), (128, 128)]), (48, 22528, 5120, 0, [(64, 128), (128, 128)]), (33, 22528, 5120, 0, [(64, 128), (128, 128)]),
    (63, 27648, 13824, 0, [(64, 128), (128, 128)]), (128, 11264, 13824, 1, [(64, 128)]), (128, 13824, 5120, 1, [(64, 128)]),
    (33, 27648, 8192, 0, [(64, 64)]), (33, 27648, 768, 0, [(64, 64)]), (2048, 2048, 8192, 0, [(128, 128)]), (8192, 8192, 8192, 0, [(256, 256)])])
def test_tiles_of_products_with_few_rows(lib, M, N, K, gated, ahead):
    rows, columns, slabs = c_int(), c_int(), c_int()
    lib.tl_gemm_direct_choice(c_int(M), c_int(N), c_int(K), c_int(gated), ctypes.byref(rows), ctypes.byref(columns), ctypes.byref(slabs))
    assert (rows.value, columns.value) in ahead
