"""float32 products at the limits of the pass that cuts the operands into heads and tails: what is taken (host only), and
operands that take several launches of it."""
import ctypes
import importlib

import pytest
import torch

from tritonix_amd import _C

mm = importlib.import_module("tritonix_amd.ops.matmul")


def _status(layout, m, n, k):
    """What tnx_gemm_f32 says of the built-in choice's tile, short of launching: E_WORKSPACE (no scratch given) if it takes it."""
    lib = _C.load()
    g = _C.GemmArgs()
    g.m, g.n, g.k = m, n, k
    g.stride_am, g.stride_ak = (1, m) if layout == "tn" else (k, 1)
    g.stride_bk, g.stride_bn = (1, k) if layout == "nt" else (n, 1)
    g.stride_cm, g.stride_cn = n, 1
    g.in_dtype = g.out_dtype = _C.F32
    assert lib.tnx_gemm_default_config(ctypes.byref(g)) == _C.OK
    g.a = g.b = g.c = 1 << 20                                    # never dereferenced
    g.workspace, g.workspace_bytes = 1 << 20, 1 << 40
    return lib.tnx_gemm_f32(ctypes.byref(g), None, 0)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_large_operands_are_taken(layout):
    """More than 2^34 elements, rows longer than a lane's 32-bit offset covers on the larger tiles, the largest int32 sizes."""
    for m, n, k in ((2048, 256, 9_000_000), (4096, 4096, 4_300_000), (4096, 4096, 6_000_000), (512, 512, 8_600_000), (300_000, 64, 60_000),
                    (64, 4_000_000, 4500), (2 ** 31 - 1, 1, 4), (1, 2 ** 31 - 1, 4), (1, 1, 715_000_000)):
        assert _status(layout, m, n, k) == _C.E_WORKSPACE, (m, n, k)
    assert _status(layout, 1, 1, 720_000_000) == _C.E_UNSUPPORTED          # three terms of it are past int32


@pytest.mark.gpu
@pytest.mark.parametrize("side", ["rows_of_a", "planes_of_b", "planes_of_a", "rows_of_b"])
@pytest.mark.parametrize("tile", ["pairs", "three_copies"])
def test_operands_cut_in_several_launches(side, tile, device):
    """1.23e9 elements against the launch's 2^30: results from both sides of the seam, each against float64.  Bound: three of
    four terms, 2^-16 per product, and the fp32 sum."""
    long, k, few = 300_000, 4096, 8
    cfg = dict(block_m=64, block_n=64, block_k=64, group_m=8, num_stages=4, num_warps=4) if tile == "pairs" else \
        dict(block_m=128, block_n=128, block_k=64, group_m=8, num_stages=2, num_warps=4)
    gen = torch.Generator(device).manual_seed(11)
    rows = side.startswith("rows")
    big = torch.empty((long, k) if rows else (k, long), device=device).normal_(generator=gen)
    small = torch.empty((few, k), device=device).normal_(generator=gen)
    a, b = {"rows_of_a": (big, small.t()), "planes_of_b": (small, big), "planes_of_a": (big.t(), small.t().contiguous()),
            "rows_of_b": (small, big.t())}[side]
    c = mm._launch_matmul(a, b, cfg)
    at = torch.tensor([0, 1, 65535, 131071, 262143, 262144, 262145, long - 1], device=device)
    x = (big[at] if rows else big[:, at].t()).double()
    ref, mag = x @ small.double().t(), x.abs() @ small.double().abs().t()
    got = (c[at] if side.endswith("a") else c[:, at].t()).double()
    assert bool(((got - ref).abs() <= (2.0 ** -16 + k * 2.0 ** -24) * mag).all())
