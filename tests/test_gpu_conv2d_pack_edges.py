"""The pass that packs conv2d's operands where its runs of eight elements would leave the input or its row: planes of fewer than
eight elements at the end of the input, padding before its first element, rows shorter and longer than a run at steps of 1, 2 and 3,
channel groups that end early or, in blocks of 32, do not exist.  Operands are small integers and sums stay below 2^24: every
16-bit and float32 product and sum is exact, so the result is the float64 convolution rounded once (float32: exactly it)."""
import ctypes

import pytest
import torch

from tritonix_amd import _C

pytestmark = pytest.mark.gpu

# n, c_in, h, w, c_out, r, s, stride, padding
CASES = {
    "plane_of_1": (1, 65, 1, 1, 24, 3, 3, (1, 1), (1, 1)),
    "plane_of_4": (2, 33, 2, 2, 24, 3, 3, (1, 1), (1, 1)),
    "plane_of_6_flat": (3, 40, 2, 3, 17, 1, 3, (1, 1), (0, 1)),
    "padding_first": (1, 48, 3, 2, 24, 3, 5, (1, 1), (1, 4)),
    "step_2_short_rows": (3, 136, 7, 7, 40, 1, 1, (2, 2), (0, 0)),
    "step_2_rows_of_9": (2, 129, 5, 9, 40, 1, 1, (2, 2), (0, 0)),
    "step_2_rows_of_17_padded": (2, 136, 4, 17, 24, 1, 1, (1, 2), (1, 1)),
    "step_2_rows_of_7_padded": (2, 136, 4, 7, 24, 1, 1, (1, 2), (0, 3)),
    "step_3": (2, 136, 7, 23, 24, 1, 1, (3, 3), (0, 1)),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_runs_at_the_edges(name, dtype, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    n, c, h, w, k, r, s, stride, padding = CASES[name]
    a = _C.Conv2dArgs()
    a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = n, c, h, w, k, r, s
    (a.stride_h, a.stride_w), (a.pad_h, a.pad_w), (a.dil_h, a.dil_w) = stride, padding, (1, 1)
    a.dtype = {torch.bfloat16: _C.BF16, torch.float16: _C.F16, torch.float32: _C.F32}[dtype]
    a.out_f32 = dtype == torch.float32
    need = _C.load().tnx_conv2d_packed_info(ctypes.byref(a), 0, 1, None)
    assert need > 0
    g = torch.Generator().manual_seed(len(name))
    x = torch.randint(-8, 9, (n, c, h, w), generator=g)
    wt = torch.randint(-4, 5, (k, c, r, s), generator=g)
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
