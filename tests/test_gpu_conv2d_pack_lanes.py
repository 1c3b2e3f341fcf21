"""How the pass that packs conv2d's operands deals column chunks and channel groups to lanes: 64 chunks of a single channel group or
8 of 8 groups, at counts of chunks on either side of a whole wave and workgroup.  Operands are small integers and sums stay below
2^24: every 16-bit and float32 product and sum is exact, so the result is the float64 convolution rounded once."""
import ctypes

import pytest
import torch

from tritonix_amd import _C

pytestmark = pytest.mark.gpu

CODES = {torch.bfloat16: _C.BF16, torch.float16: _C.F16, torch.float32: _C.F32}
# n, h, w, filter, stride: rows x chunks of 1, 7, 8, 9, 63, 64, 65, 255, 256, 257 and 1025 column chunks
PLANES = [(1, 1, 8, 1, 1), (7, 1, 5, 1, 1), (1, 4, 16, 1, 1), (3, 3, 7, 1, 1), (3, 7, 20, 1, 1), (4, 16, 8, 1, 1), (5, 13, 8, 1, 1), (3, 17, 35, 1, 1),
          (4, 16, 28, 1, 1), (1, 257, 4, 1, 1), (25, 41, 3, 1, 1), (3, 9, 11, 3, 1), (5, 13, 15, 3, 2), (2, 33, 31, 1, 2)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("c_in", [1, 3, 4, 5, 7, 8, 9, 17])
def test_chunks_and_groups(c_in, dtype, device):
    lib = _C.load()
    for n, h, w, f, stride in PLANES:
        a = _C.Conv2dArgs()
        a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = n, c_in, h, w, 24, f, f
        a.stride_h = a.stride_w = stride
        a.pad_h = a.pad_w = f // 2
        a.dil_h = a.dil_w = 1
        a.dtype, a.out_f32 = CODES[dtype], dtype == torch.float32
        need = lib.tnx_conv2d_packed_info(ctypes.byref(a), 0, 1, None)
        if not need:                                       # (16-bit 1x1 layers of unit stride are GEMMs)
            assert f == 1 and stride == 1 and dtype != torch.float32
            continue
        g = torch.Generator().manual_seed(n * 100 + w)
        x, wt = torch.randint(-8, 9, (n, c_in, h, w), generator=g), torch.randint(-4, 5, (24, c_in, f, f), generator=g)
        ref = torch.nn.functional.conv2d(x.double(), wt.double(), None, stride, f // 2)
        held = torch.full((64 + x.numel() + 64,), float("nan"), dtype=dtype, device=device)
        held[64:64 + x.numel()] = x.flatten().to(device, dtype)
        xd, wd = held[64:64 + x.numel()], wt.to(device, dtype)
        out = torch.full(ref.shape, float("nan"), dtype=dtype, device=device)
        ws = torch.full((need // 4 + 64,), float("nan"), dtype=torch.float32, device=device)
        a.input, a.weight, a.output = xd.data_ptr(), wd.data_ptr(), out.data_ptr()
        a.workspace, a.workspace_bytes = ws.data_ptr(), need
        a.stream = torch.cuda.current_stream().cuda_stream
        assert lib.tnx_conv2d_packed_forward(ctypes.byref(a), 0, 1) == _C.OK
        assert torch.equal(out.cpu(), ref.to(dtype)), (n, h, w, f, stride)
