"""CPU: shapes whose launch would hold 2^32 threads or more are refused on the host (past that a launch wraps without
an error and leaves the rest undone)."""
import ctypes

import pytest

from kerneldev_amd import _lib


@pytest.mark.parametrize("pack,d,Dp,T", [(True, 16, 64, 1 << 29), (True, 64, 192, 1 << 28), (False, 64, 256, 1 << 29)])
def test_x3_rows(pack, d, Dp, T):
    lib, a = _lib.load(), _lib.X3Args()
    a.n, a.B, a.H, a.T, a.d, a.Dp = 1, 1, 1, T, d, Dp
    a.src[0], a.lo[0], a.dst[0], a.sel[0] = 4096, 4096, 4096, 1
    for st in (a.src_strides[0], a.dst_strides[0]):
        st[0], st[1], st[2] = T * d, T * d, d
    fn = lib.kd_x3_pack if pack else lib.kd_x3_unpack
    assert fn(ctypes.byref(a), None) == _lib.KD_ERR_UNSUPPORTED
    assert "rows" in lib.kd_last_error_string().decode()


def test_span_count_rows():
    lib, a = _lib.load(), _lib.SpanArgs()
    a.tokens, a.B, a.T = 4096, 1 << 26, 1
    assert lib.kd_span_count(ctypes.byref(a), ctypes.c_void_p(4096), None) == _lib.KD_ERR_UNSUPPORTED
