"""float32 products on the binary32 matrix instruction (the block_k = 32 tiles of tnx_gemm_f32), against the float64 product, and
the choices by modelled time: every one of them has a kernel that takes the problem."""
import ctypes
import random

import pytest
import torch

from tritonix_amd import _C
import importlib

mm = importlib.import_module("tritonix_amd.ops.matmul")
TILES = ((32, 64, 4, 4), (64, 64, 4, 4), (32, 128, 4, 3))


def _args(dt, layout, m, n, k):
    g = _C.GemmArgs()
    g.m, g.n, g.k = m, n, k
    g.stride_am, g.stride_ak = (1, m) if layout == "tn" else (k, 1)
    g.stride_bk, g.stride_bn = (1, k) if layout == "nt" else (n, 1)
    g.stride_cm, g.stride_cn = n, 1
    g.in_dtype, g.out_dtype = dt, _C.I32 if dt == _C.I8 else dt
    return g


def test_priced_choices_have_kernels():
    lib, rng = _C.load(), random.Random(5)
    direct = 0
    for _ in range(1500):
        size = lambda lo, hi: int(round(lo * (hi / lo) ** rng.random()))          # noqa: E731
        dt, layout = rng.choice((_C.BF16, _C.F16, _C.I8, _C.F32)), rng.choice(("nn", "nt", "tn"))
        g = _args(dt, layout, size(16, 8192), size(16, 28672), size(16, 14336))
        if dt == _C.F32:
            assert lib.tnx_gemm_f32_config(ctypes.byref(g)) == _C.OK
            if g.block_k == 32:
                direct += 1
                assert lib.tnx_gemm_f32_scratch_bytes(ctypes.byref(g)) == 0
        else:
            assert lib.tnx_gemm_default_config(ctypes.byref(g)) == _C.OK
            st = lib.tnx_gemm_supported(ctypes.byref(g))
            assert st == _C.OK, (dt, layout, g.m, g.n, g.k, g.block_m, g.block_n, g.split_k)
        if g.split_k > 1:
            kt = -(-g.k // (32 if g.block_k == 32 else g.block_k))
            assert g.split_k <= max(1, kt) and g.tail_tiles * g.split_k <= 512
            assert lib.tnx_gemm_workspace_bytes(ctypes.byref(g)) <= (64 << 20) + 65536
    assert direct > 100


def test_where_the_operands_stay_as_they_are():
    lib = _C.load()

    def direct(layout, m, n, k):
        g = _args(_C.F32, layout, m, n, k)
        assert lib.tnx_gemm_f32_config(ctypes.byref(g)) == _C.OK
        return g.block_k == 32

    for layout in ("nn", "nt", "tn"):
        assert direct(layout, 8, 4096, 4096) and direct(layout, 64, 8192, 4096) and direct(layout, 256, 256, 256)
        assert not direct(layout, 2048, 2048, 2048) and not direct(layout, 4096, 4096, 1024)
    g = _args(_C.F32, "nn", 16, 512, 512)
    g.stride_am, g.stride_ak = 1024, 2                       # neither dimension contiguous
    assert lib.tnx_gemm_f32_config(ctypes.byref(g)) == _C.OK and g.block_k != 32
    g = _args(_C.F32, "nn", 16, 512, 0)
    assert lib.tnx_gemm_f32_config(ctypes.byref(g)) == _C.OK and g.block_k != 32
    g = _args(_C.F32, "nn", 64, 64, 64)                      # never for tnx_gemm
    g.block_m, g.block_n, g.block_k, g.num_warps, g.num_stages, g.split_k, g.group_m = 32, 64, 32, 4, 4, 1, 8
    assert lib.tnx_gemm_supported(ctypes.byref(g)) != _C.OK


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("tile", TILES)
def test_against_float64(tile, layout, device):
    """Sums of k binary32 products: k * 2^-24 of the magnitudes at the very most; edges of tiles, chunks, slabs and cuts."""
    bm, bn, nw, st = tile
    gen = torch.Generator(device).manual_seed(bm + bn)
    for m, n, k, cut in ((1, 64, 32, 1), (bm, bn, 64, 1), (bm + 1, bn - 1, 33, 1), (3, 5, 7, 1), (2 * bm - 3, 2 * bn + 5, 301, 1), (17, 130, 1000, 4),
                         (bm + 5, 3 * bn, 545, 3), (31, 4, 32 * 8, 8), (70, 66, 31, 1)):
        a = torch.randn((k, m), generator=gen, device=device).t() if layout == "tn" else torch.randn((m, k), generator=gen, device=device)
        b = torch.randn((n, k), generator=gen, device=device).t() if layout == "nt" else torch.randn((k, n), generator=gen, device=device)
        cfg = dict(block_m=bm, block_n=bn, block_k=32, group_m=8, num_stages=st, num_warps=nw)
        if cut > 1:
            cfg["split_k"] = cut
        lib = _C.load()
        g = _args(_C.F32, layout, m, n, k)
        g.block_m, g.block_n, g.block_k, g.num_warps, g.num_stages, g.split_k, g.group_m = bm, bn, 32, nw, st, cut, 8
        if lib.tnx_gemm_f32_scratch_bytes(ctypes.byref(g)) != 0:
            continue                                         # rows too short for a chunk: left to the split
        got = mm._launch_matmul(a, b, cfg)
        ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
        assert bool(((got.double() - ref).abs() <= k * 2.0 ** -24 * mag).all()), (m, n, k, cut)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_non_finite_elements_as_in_float32(layout, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    m, n, k = 20, 96, 200
    gen = torch.Generator("cpu").manual_seed(3)
    a, b = torch.randn(m, k, generator=gen), torch.randn(k, n, generator=gen)
    a[0, 0], a[1, 5], a[2, 7] = float("inf"), float("-inf"), float("nan")
    b[9, 3], b[9, 4], b[11, 5] = float("inf"), 0.0, float("nan")
    a[4, 9], a[5, 0] = 0.0, 1e-38
    x = a.t().contiguous().to(device).t() if layout == "tn" else a.to(device)
    y = b.t().contiguous().to(device).t() if layout == "nt" else b.to(device)
    got = mm.triton_matmul(x, y).cpu()
    ref = (a.double() @ b.double()).float()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    assert torch.equal(got[got.isinf()], ref[ref.isinf()])
