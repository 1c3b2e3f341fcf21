"""The pass that packs conv2d's operands at column steps of three and more (1x1 filters with such strides), and inputs of fewer
than eight elements: columns before, inside and past short rows, chunks of columns none of which the row has, channel groups that end
early.  Operands are small integers and sums stay below 2^24: every 16-bit and float32 product and sum is exact, so the result is the
float64 convolution rounded once (float32: exactly it)."""
import ctypes

import pytest
import torch

from tritonix_amd import _C

pytestmark = pytest.mark.gpu

CODES = {torch.bfloat16: _C.BF16, torch.float16: _C.F16, torch.float32: _C.F32}
# n, c_in, h, w, c_out, stride, padding
CASES = {
    "step_3": (3, 137, 9, 31, 40, (3, 3), (0, 0)),
    "step_4_long_rows": (2, 129, 5, 77, 24, (4, 4), (0, 0)),
    "step_5_padded": (2, 140, 6, 43, 24, (1, 5), (1, 4)),
    "step_7_rows_of_2": (3, 130, 5, 2, 17, (2, 7), (0, 0)),
    "step_9_padding_only_chunks": (2, 131, 3, 3, 24, (1, 9), (0, 80)),
    "step_16_one_column": (5, 33, 4, 1, 24, (3, 16), (0, 0)),
    "few_channels_step_3": (2, 3, 20, 50, 24, (3, 3), (0, 1)),
    "seven_elements_step_2": (1, 7, 1, 1, 24, (2, 2), (0, 0)),
    "six_elements_step_1": (1, 3, 1, 2, 24, (2, 1), (1, 1)),
    "four_elements_step_3": (1, 2, 1, 2, 24, (3, 3), (1, 2)),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_columns_apart(name, dtype, device):
    n, c, h, w, k, stride, padding = CASES[name]
    a = _C.Conv2dArgs()
    a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = n, c, h, w, k, 1, 1
    (a.stride_h, a.stride_w), (a.pad_h, a.pad_w), (a.dil_h, a.dil_w) = stride, padding, (1, 1)
    a.dtype, a.out_f32 = CODES[dtype], dtype == torch.float32
    need = _C.load().tnx_conv2d_packed_info(ctypes.byref(a), 0, 1, None)
    assert need > 0
    g = torch.Generator().manual_seed(len(name))
    x, wt = torch.randint(-8, 9, (n, c, h, w), generator=g), torch.randint(-4, 5, (k, c, 1, 1), generator=g)
    ref = torch.nn.functional.conv2d(x.double(), wt.double(), None, stride, padding)
    # the input between NaNs: what is read beside it must not count
    held = torch.full((64 + x.numel() + 64,), float("nan"), dtype=dtype, device=device)
    held[64:64 + x.numel()] = x.flatten().to(device, dtype)
    xd, wd = held[64:64 + x.numel()], wt.to(device, dtype)
    out = torch.full(ref.shape, float("nan"), dtype=dtype, device=device)
    ws = torch.full((need // 4 + 64,), float("nan"), dtype=torch.float32, device=device)
    a.input, a.weight, a.output = xd.data_ptr(), wd.data_ptr(), out.data_ptr()
    a.workspace, a.workspace_bytes = ws.data_ptr(), need
    a.stream = torch.cuda.current_stream().cuda_stream
    assert _C.load().tnx_conv2d_packed_forward(ctypes.byref(a), 0, 1) == _C.OK
    assert torch.equal(out.cpu(), ref.to(dtype))
