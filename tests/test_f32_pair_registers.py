"""The 256-wide float32 pair kernels keep their K loop's operands in registers: what the compiler reported of them, and their results
over every part of the loop."""
import ctypes
import json
import os

import pytest
import torch

from tritonix_amd import _C

REPORT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "build", "kernel_resources.json")


@pytest.mark.skipif(not os.path.exists(REPORT), reason="no build report (the library was built elsewhere)")
def test_spilled_registers():
    with open(REPORT) as f:
        report = json.load(f)
    pairs = {k: v["vgpr_spill"] for k, v in report.items() if k.endswith("f32 pair")}
    assert not pairs or max(pairs.values()) <= 4, {k: v for k, v in pairs.items() if v > 4}


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("cut", [1, 3])
def test_every_part_of_the_loop(layout, cut, device):
    """K of one slab (32) to several trips of the unrolled loop and each remainder, with an odd tail; rows and columns past the tile's
    end.  Three bf16 terms: 2^-16 of a product's magnitude, sums in binary32."""
    lib = _C.load()
    gen = torch.Generator(device).manual_seed(5)
    ws = torch.zeros(32 << 20, dtype=torch.uint8, device=device)
    for m, n, k in ((256, 256, 32), (257, 260, 64), (300, 511, 96), (256, 300, 129), (40, 270, 160), (513, 256, 7 * 32 + 5)):
        a = torch.randn((k, m), generator=gen, device=device).t() if layout == "tn" else torch.randn((m, k), generator=gen, device=device)
        b = torch.randn((n, k), generator=gen, device=device).t() if layout == "nt" else torch.randn((k, n), generator=gen, device=device)
        c = torch.empty(m, n, device=device)
        g = _C.GemmArgs()
        g.m, g.n, g.k = m, n, k
        (g.stride_am, g.stride_ak), (g.stride_bk, g.stride_bn), (g.stride_cm, g.stride_cn) = a.stride(), b.stride(), c.stride()
        g.in_dtype = g.out_dtype = _C.F32
        g.block_m, g.block_n, g.block_k, g.num_warps, g.num_stages, g.split_k, g.group_m = 256, 256, 64, 8, 2, cut, 8
        need = int(lib.tnx_gemm_f32_scratch_bytes(ctypes.byref(g)))
        scratch = torch.empty(need, dtype=torch.uint8, device=device)
        g.a, g.b, g.c, g.stream = a.data_ptr(), b.data_ptr(), c.data_ptr(), torch.cuda.current_stream().cuda_stream
        g.workspace, g.workspace_bytes = ws.data_ptr(), ws.numel()
        assert lib.tnx_gemm_f32(ctypes.byref(g), scratch.data_ptr(), need) == _C.OK
        mag = a.double().abs() @ b.double().abs()
        assert bool(((c.double() - a.double() @ b.double()).abs() <= (2.0 ** -16 + k * 2.0 ** -24) * mag).all()), (m, n, k)
