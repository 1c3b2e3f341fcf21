"""Slices read back by one row-block alone (eight together) and by two: every number of slices around a batch, rows on both sides of a
row-block's end, three launches over one workspace, against whole numbers."""
import ctypes

import pytest
import torch

from tritonix_amd import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("atomic", [False, True], ids=["ordered", "atomic"])
@pytest.mark.parametrize("tile", [(_C.I8, 64, 128, 128, 8, 3), (_C.BF16, 64, 128, 64, 8, 3), (_C.F16, 64, 64, 64, 4, 4), (_C.I8, 128, 128, 128, 8, 3)])
def test_whole_numbers(tile, atomic, device):
    dt, bm, bn, bk, nw, st = tile
    lib = _C.load()
    dtype = {_C.I8: torch.int8, _C.BF16: torch.bfloat16, _C.F16: torch.float16}[dt]
    gen = torch.Generator("cpu").manual_seed(bm + bn)
    ws = torch.zeros(64 << 20, dtype=torch.uint8, device=device)
    for m in (1, 15, 16, 17, 33, bm):
        for cut in (2, 7, 8, 9, 16):
            k, n = 16 * bk, bn + 24
            a, b = torch.randint(-3, 4, (m, k), generator=gen), torch.randint(-3, 4, (k, n), generator=gen)
            b[:, ::2] *= (torch.arange(k) % 8 == 0).unsqueeze(1)                    # (sums that 16 bits hold exactly)
            b[:, 1::2] *= (torch.arange(k) % 8 == 3).unsqueeze(1)
            want = (a.double() @ b.double())
            ad, bd = a.to(dtype).to(device), b.to(dtype).to(device)
            c = torch.full((m, n), -1, dtype=torch.int32 if dt == _C.I8 else dtype, device=device)
            g = _C.GemmArgs()
            g.m, g.n, g.k = m, n, k
            g.stride_am, g.stride_ak, g.stride_bk, g.stride_bn, g.stride_cm, g.stride_cn = k, 1, n, 1, n, 1
            g.in_dtype, g.out_dtype = dt, _C.I32 if dt == _C.I8 else dt
            g.block_m, g.block_n, g.block_k, g.num_warps, g.num_stages, g.split_k, g.group_m = bm, bn, bk, nw, st, cut, 8
            g.schedule = _C.SCHED_ATOMIC_REDUCE if atomic else 0
            g.a, g.b, g.c, g.stream = ad.data_ptr(), bd.data_ptr(), c.data_ptr(), torch.cuda.current_stream().cuda_stream
            if atomic:
                ws.zero_()                                                          # sums start from zero and are left so
            g.workspace, g.workspace_bytes = ws.data_ptr(), ws.numel()
            for _ in range(3):
                c.fill_(-1)
                assert lib.tnx_gemm(ctypes.byref(g)) == _C.OK, (m, cut)
                assert torch.equal(c.double().cpu(), want.to(c.dtype).double()), (m, cut)
