"""The rules by which products choose a tile, called as the host calls them."""
import ctypes
from ctypes import c_int

import pytest

from torchlet_amd.kernels import build


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(str(build.build("gemm", quiet=True)))


# 1: 64 x 64, 2: 64 x 128, 3: 128 x 128, 4: 64 x 32, 5: 32 x 32; a launch has up to 65535 rows of tiles
@pytest.mark.parametrize("M, N, want", [(65535 * 32, 32, 4), (65535 * 64, 64, 1), (65535 * 64 + 1, 32, 3), (65535 * 64 + 1, 64, 3), (65535 * 64 + 1, 192, 3), (65535 * 128, 64, 3)])
def test_32_bit_tiles_fit_a_launch(lib, M, N, want):
    assert lib.tl_gemm_f32_tile(c_int(M), c_int(N)) == want
    assert -(-M // {1: 64, 2: 64, 3: 128, 4: 64, 5: 32}[want]) <= 65535


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


# 32 bits, 2: multiply-adds, 3: matrix cores behind a copy of x, 9: rings; one and two rows stay with the multiply-adds wherever the rings, which take as long for one row as for eight, are behind
@pytest.mark.parametrize("M, N, K, want", [
    (1, 1024, 1024, 2), (1, 2048, 2048, 2), (1, 32768, 1024, 2), (1, 22016, 4096, 2), (1, 8192, 6144, 2), (1, 1536, 8192, 2), (1, 2048, 3584, 2), (1, 37888, 3584, 2), (1, 16384, 8192, 9), (1, 2560, 3584, 9), (1, 4608, 3584, 9), (1, 4096, 8192, 9),
    (1, 2048, 18944, 9), (2, 1024, 1024, 2), (2, 2048, 2048, 2), (2, 7168, 4096, 2), (2, 2560, 2560, 2), (2, 55296, 5120, 2), (2, 10240, 5120, 9), (2, 3584, 2560, 9), (2, 4608, 3584, 9), (2, 4608, 5120, 9), (2, 1024, 6848, 2),
    (3, 1024, 1024, 9), (4, 2048, 2048, 9), (8, 1000, 2048, 2), (8, 2048, 992, 2), (8, 2048, 1028, 2), (9, 64, 96, 9), (16, 4100, 1028, 3)])
def test_32_bit_products_of_few_rows_go_where_they_were_faster(lib, M, N, K, want):
    assert lib.tl_gemm_f32_few_rows_choice(c_int(M), c_int(N), c_int(K)) == want


# 0: rings of slabs, 1: the few-rows kernel that fetches into registers, 2: tiles; sizes on both sides of each line, measured 4 % and more apart
@pytest.mark.parametrize("M, N, K, gated, want", [
    (1, 32768, 768, 0, 0), (1, 152064, 3584, 0, 1), (8, 152064, 3584, 0, 0), (9, 152064, 3584, 0, 2), (16, 32768, 64, 0, 0),
    (32, 24576, 64, 0, 0), (24, 28672, 128, 0, 2), (32, 27648, 1024, 0, 2), (32, 27648, 2048, 0, 0), (17, 32832, 4096, 0, 2),
    (64, 8192, 64, 0, 0), (56, 32000, 128, 0, 2), (48, 16384, 768, 0, 2), (64, 20480, 256, 0, 2), (33, 24576, 2048, 0, 0), (64, 27648, 5120, 0, 2), (64, 29392, 6848, 0, 2), (40, 32768, 4096, 0, 0),
    (8, 20480, 256, 1, 1), (1, 20480, 768, 1, 0), (8, 20480, 1024, 1, 0), (16, 16384, 64, 1, 0), (32, 12288, 64, 1, 0), (32, 13312, 4096, 1, 2), (64, 8192, 64, 1, 0), (48, 10240, 192, 1, 2),
    (64, 12288, 1536, 1, 2), (33, 12288, 2048, 1, 0)])
def test_few_rows_go_where_they_were_faster(lib, M, N, K, gated, want):
    assert lib.tl_gemm_few_rows_choice(c_int(M), c_int(N), c_int(K), c_int(gated)) == want


# slabs of K in ranges, sizes on both sides of each line, measured 3 % and more apart
@pytest.mark.parametrize("M, N, K, want", [(32, 3072, 8192, 0), (2, 2048, 2048, 0), (33, 4096, 4096, 2), (64, 3072, 8192, 2), (48, 2048, 8192, 2), (33, 2304, 9728, 2), (64, 5120, 8192, 2), (64, 4096, 9728, 2),
                                           (64, 3584, 8192, 0), (33, 6144, 13824, 0), (64, 1536, 9728, 0), (64, 768, 27648, 0), (64, 4096, 8192, 0), (48, 2048, 16384, 0), (48, 8192, 16384, 0)])
def test_slabs_of_few_rows_come_from_what_was_faster(lib, M, N, K, want):
    assert lib.tl_gemm_slabs_choice(c_int(M), c_int(N), c_int(K)) == want


# a unit's work-groups: 4 requests twice where 8 (a gate's rows up to 8 also 6) would have it to themselves with two slabs on their way; shares of all outputs by equal numbers
@pytest.mark.parametrize("total, M, halves, even, want", [
    (16384, 1, 1, 0, (4, 32)), (14336, 16, 1, 0, (4, 28)), (12288, 8, 1, 0, (6, 48)), (8192, 2, 2, 0, (4, 16)), (5120, 8, 2, 0, (4, 10)), (5120, 9, 2, 0, (6, 20)), (8192, 16, 2, 0, (4, 16)),
    (16384, 17, 1, 0, (8, 64)), (4608, 1, 1, 1, (3, 18)), (16640, 3, 1, 0, (3, 22)), (100, 1, 1, 0, (1, 8)), (13568, 8, 1, 1, (4, 28))])
def test_shares_of_the_rings(lib, total, M, halves, even, want):
    wj, rows = c_int(), c_int()
    lib.tl_gemm_ring_plan(c_int(total), c_int(M), c_int(3584), c_int(halves), c_int(256), c_int(even), c_int(1), ctypes.byref(wj), ctypes.byref(rows))
    assert (wj.value, rows.value) == want
    assert rows.value <= 8 * wj.value // halves and (not even or rows.value % 2 == 0)


def test_shares_do_not_hang_on_the_number_of_rows_where_the_order_of_the_sums_hangs_on_the_shares(lib):
    for total in list(range(1, 3000, 97)) + list(range(3000, 40000, 523)):
        for K in (2048, 4096, 16384):
            for halves, even in ((1, 0), (1, 1), (2, 0)):
                plans = set()
                for M in range(1, 17):
                    wj, rows = c_int(), c_int()
                    lib.tl_gemm_ring_plan(c_int(total), c_int(M), c_int(K), c_int(halves), c_int(256), c_int(even), c_int(1), ctypes.byref(wj), ctypes.byref(rows))
                    plans.add((wj.value, rows.value))
                assert len(plans) == 1, (total, K, halves, even)


# 32 bits: gates and rotations by pairs of rows, also in shapes of three requests
@pytest.mark.parametrize("total, M, K, pairs, want", [(18944, 4, 3584, 1, (4, 15)), (27648, 4, 5120, 1, (6, 22)), (2304, 4, 3584, 1, (3, 9)), (3584, 8, 5120, 1, (4, 14)), (67, 4, 3584, 1, (2, 4)),
                                                      (37888, 4, 3584, 0, (4, 30)), (152064, 4, 3584, 0, (8, 60)), (3584, 4, 18944, 0, (2, 14)), (4608, 12, 3584, 0, (3, 18)), (512, 16, 512, 0, (1, 8))])
def test_shares_of_the_rings_in_32_bits(lib, total, M, K, pairs, want):
    wj, rows = c_int(), c_int()
    lib.tl_gemm_f32_ring_plan(c_int(total), c_int(M), c_int(K), c_int(pairs), c_int(256), ctypes.byref(wj), ctypes.byref(rows))
    assert (wj.value, rows.value) == want


def test_shares_in_32_bits_do_not_hang_on_the_number_of_rows_where_the_order_of_the_sums_hangs_on_the_shares(lib):
    for total in list(range(1, 3000, 97)) + list(range(3000, 40000, 523)):
        for K in (1024, 2048, 4096, 16384):
            for pairs in (0, 1):
                plans = set()
                for M in range(1, 17):
                    wj, rows = c_int(), c_int()
                    lib.tl_gemm_f32_ring_plan(c_int(total), c_int(M), c_int(K), c_int(pairs), c_int(256), ctypes.byref(wj), ctypes.byref(rows))
                    plans.add((wj.value, rows.value))
                assert len(plans) == 1, (total, K, pairs)


# ranges of K: a unit's work-group of eight requests stays alone
@pytest.mark.parametrize("total, M, K, parts, want", [(3584, 8, 18944, 4, (8, 56)), (4096, 1, 4096, 4, (8, 64)), (5120, 16, 13824, 3, (8, 61)), (2048, 8, 8192, 8, (8, 64)), (2048, 8, 2048, 4, (4, 32))])
def test_shares_of_the_rings_with_k_split(lib, total, M, K, parts, want):
    wj, rows = c_int(), c_int()
    lib.tl_gemm_ring_plan(c_int(total), c_int(M), c_int(K), c_int(1), c_int(256), c_int(0), c_int(parts), ctypes.byref(wj), ctypes.byref(rows))
    assert (wj.value, rows.value) == want


# tiles of blocks of 16 (4: 64 x 32, 5: 32 x 32) beside those of blocks of 32, sizes measured 5 % and more apart from the next
@pytest.mark.parametrize("M, N, want", [(17, 4608, 5), (33, 2052, 5), (40, 288, 5), (100, 3584, 4), (200, 2048, 4), (64, 5632, 4), (753, 3584, 1), (753, 4608, 2), (301, 37888, 2), (753, 37888, 3)])
def test_32_bit_tiles_of_small_blocks(lib, M, N, want):
    assert lib.tl_gemm_f32_tile(c_int(M), c_int(N)) == want
