"""The scratch of a float32 product is asked for before there are pointers: the answer must not depend on them."""
import ctypes

import pytest
import torch

from tritonix_amd import _C

TILES = ((32, 64, 32, 4, 4), (64, 64, 32, 4, 4), (32, 128, 32, 4, 3), (128, 128, 64, 4, 3))
# (m, n, k, stride_am, stride_ak, stride_bk, stride_bn): plain, off 16 bytes, one row for all of A, one for all of B, one column
# for all of B, rows that overlap, m-contiguous A with one plane
STRIDES = ((16, 64, 64, 64, 1, 64, 1), (16, 63, 61, 61, 1, 63, 1), (16, 64, 64, 0, 1, 64, 1), (16, 64, 64, 64, 1, 0, 1), (16, 64, 64, 64, 1, 1, 0),
           (16, 64, 64, 32, 1, 64, 1), (16, 64, 64, 1, 0, 64, 1), (16, 64, 64, 1, 16, 64, 1), (16, 64, 64, 64, 1, 1, 64))


def _args(shape, tile):
    g = _C.GemmArgs()
    g.m, g.n, g.k, g.stride_am, g.stride_ak, g.stride_bk, g.stride_bn = shape
    g.stride_cm, g.stride_cn = g.n, 1
    g.in_dtype = g.out_dtype = _C.F32
    g.block_m, g.block_n, g.block_k, g.num_warps, g.num_stages = tile
    g.split_k, g.group_m = 1, 8
    return g


@pytest.mark.parametrize("shape", STRIDES)
@pytest.mark.parametrize("tile", TILES)
def test_the_query_does_not_look_at_the_pointers(tile, shape):
    lib, asked = _C.load(), set()
    for a, b in ((None, None), (256, 512), (260, 512), (256, 516), (260, 516)):
        g = _args(shape, tile)
        g.a, g.b = a, b
        asked.add(int(lib.tnx_gemm_f32_scratch_bytes(ctypes.byref(g))))
    assert len(asked) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("shape", STRIDES)
def test_a_call_needs_what_the_query_said(shape, device):
    lib = _C.load()
    gen = torch.Generator(device).manual_seed(1)
    store = torch.randn(2, 8192, generator=gen, device=device)
    m, n, k = shape[:3]
    for tile in TILES:
        for off in (0, 1):
            a, b = (store[i, off:].as_strided((r, c), st) for i, (r, c, st) in enumerate(((m, k, shape[3:5]), (k, n, shape[5:7]))))
            g, c = _args(shape, tile), torch.empty(m, n, device=device)
            need = int(lib.tnx_gemm_f32_scratch_bytes(ctypes.byref(g)))
            scratch = torch.empty(max(need, 1), dtype=torch.uint8, device=device)
            g.a, g.b, g.c, g.stream = a.data_ptr(), b.data_ptr(), c.data_ptr(), torch.cuda.current_stream().cuda_stream
            status = lib.tnx_gemm_f32(ctypes.byref(g), scratch.data_ptr() if need else None, need)
            if status == _C.E_UNSUPPORTED:                      # no bf16 tile of these sizes for what the direct one refuses
                assert need and tile[2] == 32 and shape in STRIDES[2:7] and (off or shape[4] == 0)
                continue
            assert status == _C.OK, (tile, off, status)
            mag = a.double().abs() @ b.double().abs()           # three bf16 terms: 2^-16 of a product at most, sums in binary32
            assert bool(((c.double() - a.double() @ b.double()).abs() <= (2.0 ** -16 + k * 2.0 ** -24) * mag).all()), (tile, off)
