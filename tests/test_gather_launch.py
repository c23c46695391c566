"""CPU test of the launch rule of a single image's transposed rotation: the
angle groups minimise rounds x angles per wave, with the rounds counted in the
waves that the device really holds (one workgroup of `waves` waves a CU, less
than 16 where the LDS of n's tables and the tiles' accumulators ends)."""
import ctypes as C
import math

import pytest

from tracetransform_amd import _lib


def launch(n, A, codes, cus=256):
    w, g = C.c_int(), C.c_int()
    st = _lib.load().tt_testing_gather_launch(n, A, cus, (C.c_int32 * len(codes))(*codes),
                                              len(codes), C.byref(w), C.byref(g))
    assert st == _lib.TT_OK, _lib.load().tt_last_error()
    return w.value, g.value


@pytest.mark.parametrize("codes", [[0], [0, 3], [0, 1, 2, 3, 4, 5], list(range(8))])
def test_groups_cost_least_in_real_rounds(codes):
    for n in (3, 64, 133, 363, 521, 725, 1000, 1163, 1449, 1517, 1800):
        for A in (1, 7, 31, 90, 360, 720):
            waves, groups = launch(n, A, codes)
            assert 9 <= waves <= 16
            tiles = -(-n // 30) * -(-n // 32)

            def cost(g):
                return math.ceil(tiles * g / (256 * waves)) * math.ceil(A / g) + g * n * n / 4.2e6

            assert groups <= min(A, 32)
            assert cost(groups) == min(cost(g) for g in range(1, min(A, 32) + 1)), (n, A)


def test_no_second_round_for_a_few_waves():
    # 575 tiles, 15 waves a CU: 7 groups would be 4025 waves, 185 more than a
    # round; 20 fill three rounds to 99.8 %.  3420 tiles, 13 waves a CU: the
    # partial images of many groups cost more than fuller rounds give.
    assert launch(725, 360, list(range(8))) == (15, 20)
    assert launch(1800, 90, list(range(8))) == (13, 10)
