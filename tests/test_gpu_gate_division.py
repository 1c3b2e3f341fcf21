"""The gate of 16-bit results: the binary32 value that the float32 epilogue stores (which divides), rounded once."""
import ctypes

import pytest
import torch

from tritonix_amd import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", [_C.EPI_GLU_SILU, _C.EPI_GLU_SIGMOID])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("spread", [1.0, 12.0])
def test_bits_of_the_division(dtype, act, spread, device):
    m, n, k, lib = 4096, 2048, 64, _C.load()
    gen = torch.Generator(device).manual_seed(3)
    x = torch.randn(m, k, generator=gen, device=device).to(dtype)
    w = (torch.randn(k, n, generator=gen, device=device) * spread / 8).to(dtype)
    out = {}
    for out_dtype in (dtype, torch.float32):
        z = out[out_dtype] = torch.empty(m, n // 2, dtype=out_dtype, device=device)
        g = _C.GemmArgs()
        g.m, g.n, g.k = m, n, k
        g.stride_am, g.stride_ak, g.stride_bk, g.stride_bn, g.stride_cm, g.stride_cn = k, 1, n, 1, n // 2, 1
        g.in_dtype = {torch.float16: _C.F16, torch.bfloat16: _C.BF16}[dtype]
        g.out_dtype = _C.F32 if out_dtype == torch.float32 else g.in_dtype
        g.block_m, g.block_n, g.block_k, g.num_warps, g.num_stages = 128, 128, 64, 8, 3
        g.split_k, g.group_m, g.epilogue = 1, 8, act
        g.a, g.b, g.c, g.stream = x.data_ptr(), w.data_ptr(), z.data_ptr(), torch.cuda.current_stream().cuda_stream
        assert lib.tnx_gemm(ctypes.byref(g)) == _C.OK
    assert bool((out[torch.float32].abs() > 2.0 ** -126).float().mean() > 0.99)
    assert int((out[dtype] != out[torch.float32].to(dtype)).sum()) == 0
