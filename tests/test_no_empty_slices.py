"""Built-in K cuts: every slice of a cut tile has a K slab of its own."""
import ctypes
import random

from tritonix_amd import _C


def _empty(kt, s):
    return s > 1 and (s - 1) * -(-kt // s) >= kt


def test_products():
    lib, rng, cut = _C.load(), random.Random(8), 0
    size = lambda lo, hi: int(round(lo * (hi / lo) ** rng.random()))          # noqa: E731
    named = [(_C.I8, "nn", 691, 17, 10318), (_C.BF16, "nn", 17, 18, 9344), (_C.F16, "nt", 31, 752, 8247), (_C.I8, "tn", 48, 4096, 16 * 129)]
    drawn = [(rng.choice((_C.BF16, _C.F16, _C.I8, _C.F32)), rng.choice(("nn", "nt", "tn")), size(1, 2048), size(16, 28672), size(64, 14336))
             for _ in range(6000)]
    for dt, layout, m, n, k in named + drawn:
        g = _C.GemmArgs()
        g.m, g.n, g.k = m, n, k
        g.stride_am, g.stride_ak = (1, m) if layout == "tn" else (k, 1)
        g.stride_bk, g.stride_bn = (1, k) if layout == "nt" else (n, 1)
        g.stride_cm, g.stride_cn = n, 1
        g.in_dtype, g.out_dtype = dt, _C.I32 if dt == _C.I8 else dt
        assert (lib.tnx_gemm_f32_config if dt == _C.F32 else lib.tnx_gemm_default_config)(ctypes.byref(g)) == _C.OK
        kt = -(-k // g.block_k)
        if dt == _C.F32 and g.block_k == 64:
            kt = -(-k // 32)                                                   # heads and tails: 32 k to a slab
        cut += g.split_k > 1
        assert not _empty(kt, g.split_k), (dt, layout, m, n, k, g.split_k)
    assert cut > 1000


def test_conv2d_layers():
    lib, rng, cut = _C.load(), random.Random(9), 0
    info = (ctypes.c_int32 * 6)()
    for _ in range(4000):
        a = _C.Conv2dArgs()
        f = rng.choice((1, 3, 5))
        a.batch, a.c_in, a.c_out = rng.choice((1, 4, 8)), 8 * rng.randint(1, 48), rng.randint(16, 512)
        a.h_in = a.w_in = rng.choice((7, 14, 17, 28))
        a.filter_h = a.filter_w = f
        a.stride_h = a.stride_w = rng.choice((1, 2))
        a.pad_h = a.pad_w = f // 2
        a.dil_h = a.dil_w = 1
        a.dtype = _C.BF16
        if not lib.tnx_conv2d_packed_info(ctypes.byref(a), -1, 1, info):
            continue
        kt = -(-f * f * (a.c_in // 8) // 8)
        cut += info[4] > 1
        assert not _empty(kt, info[4]), (a.batch, a.c_in, a.c_out, a.h_in, f, info[4])
    assert cut > 200
