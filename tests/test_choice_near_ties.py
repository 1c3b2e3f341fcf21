"""Built-in tiles where the modelled times of two lie close together: the one that was measured to be faster."""
import ctypes

import pytest

from tritonix_amd import _C

# m, n, k, layout, the tile not to take (slower by 14 to 40 %)
MEASURED = [(3776, 72, 5952, "nn", (128, 64)), (3776, 72, 5952, "nt", (128, 64)), (1280, 352, 4672, "nn", (128, 64)), (1344, 288, 7136, "nn", (128, 64)),
            (1856, 704, 3320, "nn", (128, 64)), (4240, 80, 7104, "nt", (128, 64)), (1024, 13122, 64, "tn", (192, 256)), (896, 14347, 64, "nn", (192, 256)),
            (576, 5568, 512, "nn", (64, 256)), (109, 25344, 232, "nn", (64, 256))]


@pytest.mark.parametrize("dtype", [_C.BF16, _C.F16])
@pytest.mark.parametrize("m, n, k, layout, slow", MEASURED)
def test_the_slower_tile_is_not_chosen(m, n, k, layout, slow, dtype):
    g = _C.GemmArgs()
    g.m, g.n, g.k = m, n, k
    g.stride_am, g.stride_ak = (1, m) if layout == "tn" else (k, 1)
    g.stride_bk, g.stride_bn = (1, k) if layout == "nt" else (n, 1)
    g.stride_cm, g.stride_cn = n, 1
    g.in_dtype = g.out_dtype = dtype
    assert _C.load().tnx_gemm_default_config(ctypes.byref(g)) == _C.OK
    assert (g.block_m, g.block_n) != slow
