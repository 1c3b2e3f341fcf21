"""The built-in choice for few rows, on the host: where it cuts K and where it leaves the loop whole."""
import ctypes

from tritonix_amd import _C

TYPES = {"bf16": (_C.BF16, _C.BF16), "f16": (_C.F16, _C.F16), "i8": (_C.I8, _C.I32), "f32": (_C.F32, _C.F32)}


def _choice(dt, layout, m, n, k):
    g = _C.GemmArgs()
    g.m, g.n, g.k = m, n, k
    g.stride_am, g.stride_ak = (1, m) if layout == "tn" else (k, 1)
    g.stride_bk, g.stride_bn = (1, k) if layout == "nt" else (n, 1)
    g.stride_cm, g.stride_cn = n, 1
    g.in_dtype, g.out_dtype = TYPES[dt]
    assert _C.load().tnx_gemm_default_config(ctypes.byref(g)) == _C.OK
    return g


def test_a_short_loop_is_not_cut():
    """A cut that saves a slab or two of 0.1 to 0.3 us pays 1.2 to 2.5 us for handing the slices over."""
    for dt, least, slab in (("bf16", 18, 64), ("f16", 18, 64), ("i8", 12, 128), ("f32", 14, 32)):
        for layout in ("nn", "nt"):
            for m in (1, 16, 33, 64):
                for n in (64, 512, 4096, 16384):
                    for kt in range(1, least):
                        for k in (kt * slab, kt * slab - slab + 1):
                            assert _choice(dt, layout, m, n, k).split_k == 1, (dt, layout, m, n, k)
    for dt, k in (("bf16", 18 * 64), ("i8", 12 * 128), ("f32", 14 * 32)):
        assert _choice(dt, "nn", 16, 512, k).split_k >= 4


def test_long_runs_of_a_k_contiguous_b():
    assert _choice("bf16", "nt", 16, 8192, 4096).split_k == 4          # two slices of 32 slabs: one cut more
    assert _choice("bf16", "nt", 16, 8192, 8192).split_k == 2
    assert _choice("bf16", "nn", 16, 8192, 4096).split_k == 2
    assert _choice("f32", "nt", 16, 8192, 6144).split_k == 4           # two slices of 96
    assert _choice("i8", "nt", 16, 28672, 4096).split_k == 2
    assert _choice("bf16", "nt", 16, 28672, 2048).split_k == 1
    g = _choice("f32", "nt", 16, 16384, 3072)                           # 96 slabs uncut
    assert (g.block_n, g.split_k) == (128, 2) and _choice("f32", "nt", 16, 16384, 4096).block_n == 64
    assert (_choice("bf16", "nt", 16, 16384, 14336).block_n, _choice("bf16", "nt", 16, 28672, 14336).block_n) == (128, 64)


def test_every_choice_for_few_rows_is_launchable():
    lib = _C.load()
    for dt in ("bf16", "f16", "i8"):
        for layout in ("nn", "nt", "tn"):
            for m in (1, 2, 16, 17, 32, 33, 48, 64):
                for n in (64, 130, 1024, 8192, 28672):
                    for k in (64, 65, 640, 1024, 2048, 4096, 8192, 14336):
                        g = _choice(dt, layout, m, n, k)
                        assert lib.tnx_gemm_supported(ctypes.byref(g)) == _C.OK, (dt, layout, m, n, k)
                        assert g.split_k <= max(1, -(-k // g.block_k) // 2)


def test_int8_with_a_column_major_a():
    """128-row tiles, K cut as the row-major choice cuts it; ragged rows are copied by the wrappers."""
    import importlib

    import torch

    mm = importlib.import_module("tritonix_amd.ops.matmul")
    for m, n, k, split in ((16, 4096, 4096, 8), (48, 8192, 4096, 4), (64, 512, 14336, 16), (16, 28672, 4096, 1), (48, 4096, 1536, 1)):
        g = _choice("i8", "tn", m, n, k)
        assert (g.block_m, g.block_n, g.num_warps, g.num_stages, g.split_k) == (128, 128, 8, 3, split), (m, n, k)
    b = torch.zeros(256, 64, dtype=torch.int8)
    for m, pitch, in_place in ((16, 16, True), (64, 64, True), (16, 24, False), (15, 16, False), (40, 48, False), (65, 65, False),
                               (191, 191, False), (100, 100, True), (193, 193, True)):
        a = torch.zeros(256, pitch, dtype=torch.int8)[:, :m].t()
        x, _, layout = mm.engine_operands(a, b)
        assert (x is a) == in_place and (layout in (5, 6)) == in_place, (m, pitch)
    a = torch.zeros(256, 15, dtype=torch.bfloat16).t()
    assert mm.engine_operands(a, b.bfloat16())[0] is a
