"""Every tile of the grid is computed once in whatever order a workgroup finds it: groups of rows that do not divide the tiles, of one
row, larger than the grid, up to the largest int32; tiles cut along K, all of them and the last ones only.  (Several problems in one
grid: test_several_problems.py.)

int8 products are exact, so every comparison is for equality with the int64 product."""
import ctypes

import pytest
import torch

from tritonix_amd import _C

pytestmark = pytest.mark.gpu


def _args(a, b, c, group, split=1, tail=0, bm=64, bn=128):
    g = _C.GemmArgs()
    (g.m, g.k), g.n = a.shape, b.shape[1]
    g.a, g.b, g.c = a.data_ptr(), b.data_ptr(), c.data_ptr()
    g.stride_am, g.stride_ak = a.stride()
    g.stride_bk, g.stride_bn = b.stride()
    g.stride_cm, g.stride_cn = c.stride()
    g.in_dtype, g.out_dtype = _C.I8, _C.I32
    g.block_m, g.block_n, g.block_k, g.num_warps, g.num_stages = bm, bn, 128, 8, 3
    g.group_m, g.split_k, g.tail_tiles = group, split, tail
    g.stream = torch.cuda.current_stream().cuda_stream
    return g


@pytest.mark.parametrize("layout", ["nn", "nt"])
@pytest.mark.parametrize("m, n, k", [(64, 64, 128), (700, 330, 256), (65, 1030, 384), (1100, 64, 512)])
def test_each_tile_once(m, n, k, layout, device):
    gen = torch.Generator().manual_seed(m + n)
    a = torch.randint(-127, 128, (m, k), generator=gen, dtype=torch.int8)
    b = torch.randint(-127, 128, (n, k) if layout == "nt" else (k, n), generator=gen, dtype=torch.int8)
    b = b.t() if layout == "nt" else b
    want = (a.double() @ b.double()).to(torch.int32)
    ad, bd = a.to(device), b.to(device)
    lib = _C.load()
    for group in (1, 2, 3, 8, 17, 2 ** 31 - 1):
        for split, tail in ((1, 0), (2, 0), (3, 1), (2, 5)):
            c = torch.full((m, n), -7, dtype=torch.int32, device=device)
            g = _args(ad, bd, c, group, split, tail)
            ws = torch.zeros(max(int(lib.tnx_gemm_workspace_bytes(ctypes.byref(g))), 256), dtype=torch.uint8, device=device)
            g.workspace, g.workspace_bytes = ws.data_ptr(), ws.numel()
            for _ in range(2):                                # counters are back at zero after the first
                assert lib.tnx_gemm(ctypes.byref(g)) == _C.OK
            assert torch.equal(c.cpu(), want), (group, split, tail)


def test_rows_of_the_result_apart(device):
    """Strides of the result that 32 bits hold in elements but not in bytes, and the columns of a transposed result."""
    gen = torch.Generator().manual_seed(1)
    a, b = (torch.randint(-127, 128, s, generator=gen, dtype=torch.int8) for s in ((3, 128), (128, 80)))
    want = (a.double() @ b.double()).to(torch.int32)
    for c in (torch.zeros(2 * 300_000_000 + 80, dtype=torch.int32, device=device).as_strided((3, 80), (300_000_000, 1)),
              torch.zeros(80, 3, dtype=torch.int32, device=device).t()):
        assert _C.load().tnx_gemm(ctypes.byref(_args(a.to(device), b.to(device), c, 8))) == _C.OK
        assert torch.equal(c.cpu(), want)
