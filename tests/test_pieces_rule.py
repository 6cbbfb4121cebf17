"""CPU: where the attention lists are cut into pieces (kd_attn_*_ws_bytes, split_pieces).

Shapes timed uncut and cut on an MI355X: those that cutting slowed stay whole (the first
five were cut, and 1.1 to 1.4 times slower for it), those that it speeds up are cut."""
import ctypes

import pytest

from kerneldev_amd import _lib

BF, F32, UNEVEN, FULL = _lib.KD_BF16, _lib.KD_F32, _lib.KD_LISTS_UNEVEN, _lib.KD_LISTS_FULL


def _bytes(B, H, T, D, dtype, lists):
    lib, a = _lib.load(), _lib.AttnArgs()
    a.B, a.H, a.T, a.D, a.sm_scale, a.dtype, a.lists = B, H, T, D, D ** -0.5, dtype, lists
    return lib.kd_attn_fwd_ws_bytes(ctypes.byref(a)), lib.kd_attn_bwd_ws_bytes(ctypes.byref(a))


@pytest.mark.parametrize("shape,dtype,lists", [
    ((1, 12, 1400, 128), BF, FULL),    # dK/dV 53 us whole, 76 cut in two
    ((1, 17, 1400, 256), BF, FULL),    # forward 79, 99
    ((1, 16, 2048, 64), BF, UNEVEN),   # dQ 36, 41
    ((1, 32, 512, 64), F32, UNEVEN),   # forward 29, 35 in four
    ((2, 8, 4096, 256), F32, UNEVEN),  # 1364, 1435
    ((2, 8, 4096, 128), F32, FULL),    # 1152, 1172
    ((4, 8, 395, 128), BF, UNEVEN),
    ((8, 16, 2048, 64), BF, UNEVEN),
    ((1, 12, 5942, 256), BF, UNEVEN),  # 324, 418 in three
])
def test_shapes_that_stay_whole(shape, dtype, lists):
    assert _bytes(*shape, dtype, lists) == (0, 0)


@pytest.mark.parametrize("shape,dtype,lists", [
    ((1, 8, 4095, 128), BF, UNEVEN),   # forward 96, 77
    ((1, 1, 8192, 64), BF, FULL),      # 132, 44
    ((1, 12, 1531, 64), BF, UNEVEN),   # 37, 28
    ((2, 8, 4096, 128), F32, UNEVEN),  # 647, 625
    ((1, 2, 300, 64), F32, FULL),      # 18, 12
])
def test_shapes_that_are_cut(shape, dtype, lists):
    f, b = _bytes(*shape, dtype, lists)
    rows = shape[0] * shape[1] * shape[2]
    assert f % (4 * rows * (shape[3] + 2)) == 0 and 2 <= f // (4 * rows * (shape[3] + 2)) <= 6
    assert b > 0
