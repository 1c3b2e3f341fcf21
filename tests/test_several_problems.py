"""Several problems in one grid, and a bias per row: conv2d's 1x1 layers, one GEMM with a problem per image.

Operands are small integers: every product and sum is exact in fp32, so the result is the float64 one rounded once."""
import ctypes

import pytest
import torch

from tritonix_amd import _C
from tritonix_amd.ops.conv2d import conv2d_forward

CODES = {torch.bfloat16: _C.BF16, torch.float16: _C.F16, torch.float32: _C.F32}
# one input channel on planes of one pixel: the plane's stride of 1 makes B count as k-contiguous
NARROW = [(1, 1, 1), (4, 1, 1), (128, 1, 1), (4, 2, 1), (4, 1, 2), (3, 65, 1), (2, 64, 1), (5, 8, 3)]


def _args(n, c, hw, k, dtype=torch.bfloat16):
    a = _C.Conv2dArgs()
    a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = n, c, hw, hw, k, 1, 1
    a.stride_h = a.stride_w = a.dil_h = a.dil_w = 1
    a.dtype = CODES[dtype]
    return a


@pytest.mark.skipif(torch.cuda.is_available(), reason="host memory in the place of the operands: only where nothing can be launched")
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("n, c, hw", NARROW)
def test_what_is_supported_reaches_the_runtime(n, c, hw, bias):
    lib, held = _C.load(), ctypes.create_string_buffer(4096 + 256)
    at = (ctypes.addressof(held) + 255) // 256 * 256
    for k in (1, 24, 64, 320):
        a = _args(n, c, hw, k)
        a.input = a.weight = a.output = at
        if bias:
            a.bias, a.bias_dtype = at, _C.BF16
        assert lib.tnx_conv2d_supported(ctypes.byref(a)) == _C.OK
        status = lib.tnx_conv2d_forward(ctypes.byref(a))
        assert status == _C.OK or lib.tnx_last_hip_error() != 1, "refused as an invalid value before the launch"


def _problem(n, c, hw, k, dtype, bias_dtype, device):
    g = torch.Generator().manual_seed(n * 1000 + c * 10 + hw)
    x = torch.randint(-4, 5, (n, c, hw, hw), generator=g)
    w = torch.randint(-1, 2, (k, c, 1, 1), generator=g)
    b = torch.randint(-8, 9, (k,), generator=g) if bias_dtype else None
    ref = torch.nn.functional.conv2d(x.double(), w.double(), b.double() if b is not None else None)
    return x.to(device, dtype), w.to(device, dtype), b.to(device, bias_dtype) if b is not None else None, ref


@pytest.mark.gpu
@pytest.mark.parametrize("bias_dtype", [None, torch.float32, "own"], ids=["none", "f32", "own"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("n, c, hw", NARROW)
def test_narrow_layers(n, c, hw, dtype, bias_dtype, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    for k in (1, 24, 64, 320):
        x, w, b, ref = _problem(n, c, hw, k, dtype, dtype if bias_dtype == "own" else bias_dtype, device)
        for _ in range(2):                                  # the ordinary path, then the kept launch
            assert torch.equal(conv2d_forward(x, w, b).cpu(), ref.to(dtype)), (n, c, hw, k)


@pytest.mark.gpu
@pytest.mark.parametrize("out_f32", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_every_tile_that_takes_several_problems(dtype, out_f32, device):
    lib, taken = _C.load(), 0
    tiles = sorted({tuple(int(v) for v in name.split()[1:4]) for name in _C.kernel_names() if name.split()[0] == {torch.bfloat16: "bf16", torch.float16: "f16"}[dtype]})
    for n, c, hw, k in ((1, 72, 5, 40), (3, 72, 5, 40), (7, 64, 4, 129), (2, 40, 13, 300), (3, 1, 1, 70)):
        for bias_dtype in (None, dtype, torch.float32):
            x, w, b, ref = _problem(n, c, hw, k, dtype, bias_dtype, device)
            for bm, bn, bk in tiles:
                a = _args(n, c, hw, k, dtype)
                a.block_cout, a.block_pixels, a.block_k, a.loader, a.out_f32 = bm, bn, bk, _C.CONV_LOADER_GEMM, out_f32
                if lib.tnx_conv2d_supported(ctypes.byref(a)) != _C.OK:
                    continue
                out = torch.full(ref.shape, float("nan"), dtype=torch.float32 if out_f32 else dtype, device=device)
                a.input, a.weight, a.output = x.data_ptr(), w.data_ptr(), out.data_ptr()
                if b is not None:
                    a.bias, a.bias_dtype = b.data_ptr(), CODES[bias_dtype]
                a.stream = torch.cuda.current_stream().cuda_stream
                assert lib.tnx_conv2d_forward(ctypes.byref(a)) == _C.OK, (n, c, hw, k, bm, bn, bk)
                assert torch.equal(out.cpu(), ref.to(out.dtype)), (n, c, hw, k, bm, bn, bk, bias_dtype)
                taken += 1
    assert taken >= 5 * 3 * 5
