"""Packed conv2d tiles: a last round of a few more workgroups than CUs costs what two on a CU cost, also after whole rounds."""
import ctypes

import pytest

from tritonix_amd import _C


@pytest.mark.parametrize("dtype", [_C.BF16, _C.F16])
@pytest.mark.parametrize("layer, tile, slow", [((64, 256, 62, 28, 5, 1), 57, 75), ((64, 256, 64, 28, 5, 1), 57, 73), ((64, 384, 51, 28, 5, 1), 80, 102),
                                               ((16, 128, 37, 56, 5, 1), 40, 46)])
def test_long_tiles_where_short_ones_leave_a_remainder(layer, tile, slow, dtype):
    """784 tiles of 64x64 on 512 places leave 272 for 256 CUs; 196 of 64x256 are one round (measured: `tile` and `slow` us)."""
    n, c, k, hw, f, stride = layer
    a = _C.Conv2dArgs()
    a.batch, a.c_in, a.c_out, a.h_in, a.w_in, a.filter_h, a.filter_w = n, c, k, hw, hw, f, f
    a.stride_h = a.stride_w = stride
    a.pad_h = a.pad_w = f // 2
    a.dil_h = a.dil_w = 1
    a.dtype = dtype
    info = (ctypes.c_int32 * 6)()
    assert _C.load().tnx_conv2d_packed_info(ctypes.byref(a), -1, 1, info) > 0
    assert tuple(info[:2]) == (64, 256), list(info)
