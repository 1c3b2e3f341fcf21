"""The last K slab of operands that no tile divides: its chunks are fetched together, those that cross the end of the matrix's last
row moved back and shifted, what lies past k cleared.  Remainders of k on either side of a chunk, of n and m inside one, rows off
16 bytes, for each layout and element size, whole and with K cut, rows one after another and apart.  Small integers: sums below 2^24 are exact, so the result is the
float64 product rounded once (int8: the integer)."""
import ctypes

import pytest
import torch

from tritonix_amd import _C
from tritonix_amd.kernel import out_dtype_for

pytestmark = pytest.mark.gpu

SIZES = [(70, 130, 191), (65, 72, 129), (129, 67, 72), (33, 200, 137), (64, 64, 65), (17, 33, 1000), (200, 139, 311), (1, 9, 90), (130, 261, 127)]
TILES = {16: [(32, 64, 64, 4, 4), (64, 128, 64, 8, 3), (192, 192, 64, 8, 3), (256, 256, 64, 4, 2), (256, 256, 64, 8, 2)],
         8: [(32, 128, 128, 4, 3), (64, 128, 128, 8, 3), (192, 192, 128, 8, 3), (256, 256, 128, 4, 2), (256, 256, 128, 8, 2)]}
CODES = {torch.bfloat16: _C.BF16, torch.float16: _C.F16, torch.int8: _C.I8}


def _held(t, gap, device):
    """The matrix in the middle of a buffer of NaNs (int8: of 127), `gap` of them behind every row but the last."""
    fill = 127 if t.dtype == torch.int8 else float("nan")
    rows, cols = t.shape
    buf = torch.full((rows * (cols + gap) - gap + 256,), fill, dtype=t.dtype, device=device)
    view = buf[128:].as_strided((rows, cols), (cols + gap, 1))
    view.copy_(t.to(device))
    return view


def _built(dtype, layout):
    """The tiles of the list that have a ring loader for the layout: all but for an m-contiguous A, which some are not built for."""
    name = {torch.bfloat16: "bf16", torch.float16: "f16", torch.int8: "i8"}[dtype]
    at = {tuple(int(v) for v in k.split()[1:6]) for k in _C.kernel_names() if k.split()[0] == name and "at" in k.split()}
    return [t for t in TILES[8 if dtype == torch.int8 else 16] if layout != "tn" or t in at]


@pytest.mark.parametrize("gap", [0, 5], ids=["dense", "apart"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.int8], ids=["bf16", "f16", "i8"])
def test_last_slab(dtype, layout, gap, device):
    lib, tiles = _C.load(), _built(dtype, layout)
    taken = 0
    for m, n, k in SIZES:
        g = torch.Generator().manual_seed(m * n + k)
        a, b = torch.randint(-8, 9, (m, k), generator=g), torch.randint(-4, 5, (k, n), generator=g)
        ref = a.double() @ b.double()
        da = _held((a.t() if layout == "tn" else a).contiguous().to(dtype), gap, device)
        db = _held((b.t() if layout == "nt" else b).contiguous().to(dtype), gap, device)
        da, db = da.t() if layout == "tn" else da, db.t() if layout == "nt" else db
        for bm, bn, bk, nw, st in tiles:
            for cut in (1, 2):
                out = torch.full((m, n), 77, dtype=out_dtype_for(dtype), device=device)
                p = _C.GemmArgs()
                p.a, p.b, p.c = da.data_ptr(), db.data_ptr(), out.data_ptr()
                p.m, p.n, p.k = m, n, k
                p.stride_am, p.stride_ak = da.stride()
                p.stride_bk, p.stride_bn = db.stride()
                p.stride_cm, p.stride_cn = out.stride()
                p.in_dtype = CODES[dtype]
                p.out_dtype = _C.I32 if dtype == torch.int8 else CODES[dtype]
                p.block_m, p.block_n, p.block_k, p.num_warps, p.num_stages = bm, bn, bk, nw, st
                p.group_m, p.split_k, p.stream = 8, cut, torch.cuda.current_stream().cuda_stream
                if lib.tnx_gemm_tail_slabs(ctypes.byref(p)) != 1:
                    assert (m, layout, gap) == (1, "tn", 0)                 # one row, dense: its k is contiguous too
                    continue
                need = lib.tnx_gemm_workspace_bytes(ctypes.byref(p))
                ws = torch.zeros(max(need, 1), dtype=torch.uint8, device=device)
                p.workspace, p.workspace_bytes = ws.data_ptr(), need
                assert lib.tnx_gemm(ctypes.byref(p)) == _C.OK
                assert torch.equal(out.cpu().double(), ref.to(out.dtype).double()), (m, n, k, bm, bn, cut)
                taken += 1
    assert len(tiles) >= 2 and taken == len(tiles) * 2 * (len(SIZES) - (layout == "tn" and gap == 0))
