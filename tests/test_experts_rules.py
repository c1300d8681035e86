"""The rule by which products over the experts' rows choose a kernel, called as the host calls it."""
import ctypes
from ctypes import c_int

import pytest

from torchlet_amd.kernels import build


# 0: rings of 16 weight rows and 8 slots, 1: few rows, 2 to 5: tiles, 6: rings of 32 weight rows and 16 slots.  A launch has up to 65535 tiles of slots: 52000 groups of four slots are 65000 of 16 and
# 78000 of 8
@pytest.mark.parametrize("groups, rows, K, want", [(16, 16, 2048, 0), (16, 64, 2048, 0), (16, 65, 2048, 6), (16, 192, 2048, 6), (16, 16, 1984, 1), (16, 65, 1984, 6),
                                                   (43690, 174760, 2048, 0), (43700, 174800, 2048, 6), (52000, 208000, 2048, 6)])
def test_few_slots_a_group(groups, rows, K, want):
    lib = ctypes.CDLL(str(build.build("experts", quiet=True)))
    assert lib.tl_experts_choice(c_int(groups), c_int(rows), c_int(1024), c_int(K)) == want
