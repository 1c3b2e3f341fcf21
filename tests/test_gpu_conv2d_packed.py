"""conv2d forward over packed operands (the route taken with scratch and no tile named): geometries at the edges of its
layout and tiles against the CPU convolution in float64.

Bound: products of 16-bit operands are exact in fp32 and summed in fp32, so before the one rounding the error is at most
k * 2^-24 of the sum of magnitudes, far below half a unit of the 16-bit result (2^-9 bf16, 2^-12 f16); one such unit
on top of that covers the rounding.  float32 operands: three of four terms of a bf16 head/tail split, 2^-16 per product."""
import ctypes

import pytest
import torch

from tritonix_amd import _C
from tritonix_amd.ops.conv2d import conv2d_forward

pytestmark = pytest.mark.gpu

# n, c_in, h, w, c_out, r, s, stride, padding, dilation
CASES = {
    "3x3_whole_slabs": (2, 64, 16, 16, 128, 3, 3, (1, 1), (1, 1), (1, 1)),
    "ragged_channels": (2, 117, 9, 11, 70, 3, 3, (1, 1), (1, 1), (1, 1)),
    "shortest_k": (3, 17, 12, 10, 5, 3, 3, (1, 1), (1, 1), (1, 1)),
    "plane_7x7": (9, 64, 7, 7, 200, 3, 3, (1, 1), (1, 1), (1, 1)),          # 49 pixels: chunks of 8 stop short of a plane
    "stride_2": (2, 64, 17, 15, 96, 3, 3, (2, 2), (1, 1), (1, 1)),
    "stride_3_dilated": (2, 40, 23, 19, 64, 2, 3, (3, 2), (2, 3), (2, 2)),
    "1x1_stride_2": (2, 264, 29, 31, 72, 1, 1, (2, 2), (0, 0), (1, 1)),
    "1xs_stride_2_2": (2, 96, 9, 33, 40, 1, 3, (2, 2), (0, 1), (1, 1)),
    "rx1_stride_1_3": (2, 96, 33, 9, 40, 3, 1, (1, 3), (1, 0), (1, 1)),
    "pad_wider_than_image": (1, 32, 3, 2, 24, 5, 5, (1, 1), (4, 4), (1, 1)),
    "one_output": (1, 64, 5, 5, 33, 5, 5, (1, 1), (0, 0), (1, 1)),
    "long_k_padded_table": (1, 468, 6, 6, 40, 7, 7, (1, 1), (3, 3), (1, 1)),   # offset table per slab only after rounding c_in up
    "cut_k": (1, 512, 7, 7, 512, 3, 3, (1, 1), (1, 1), (1, 1)),               # few tiles, long k: K slices meet in the workspace
    # float32: blocks of 32 channels, whole and padded, on either side of where three terms are taken instead
    "one_block": (2, 32, 9, 10, 40, 3, 3, (1, 1), (1, 1), (1, 1)),
    "block_padded": (1, 25, 12, 9, 72, 3, 3, (2, 1), (1, 1), (1, 1)),
    "three_terms_33": (2, 33, 9, 9, 24, 3, 3, (1, 1), (1, 1), (1, 1)),
    "two_blocks_padded": (2, 51, 8, 11, 130, 2, 3, (1, 2), (1, 0), (2, 1)),
    "blocks_1x1_stride_2": (3, 265, 15, 17, 64, 1, 1, (2, 2), (0, 0), (1, 1)),
    "blocks_cut_k": (1, 512, 7, 9, 300, 3, 3, (1, 1), (1, 1), (1, 1)),
    "many_tiles": (16, 64, 57, 55, 256, 3, 3, (1, 1), (1, 1), (1, 1)),
}


def _run(name, dtype, device, bias=True):
    n, c, h, w, k, r, s, stride, padding, dilation = CASES[name]
    g = torch.Generator().manual_seed(len(name))
    x = torch.randn(n, c, h, w, generator=g).to(dtype)
    wt = (torch.randn(k, c, r, s, generator=g) / (c * r * s) ** 0.5).to(dtype)
    b = torch.randn(k, generator=g).to(dtype) if bias else None
    out = conv2d_forward(x.to(device), wt.to(device), None if b is None else b.to(device), stride, padding, dilation)
    sample = slice(0, n) if n * k * h * w < 2 << 20 else slice(n - 1, n)
    b64 = None if b is None else b.double()
    ref = torch.nn.functional.conv2d(x[sample].double(), wt.double(), b64, stride, padding, dilation)
    mag = torch.nn.functional.conv2d(x[sample].double().abs(), wt.double().abs(), None if b is None else b64.abs(), stride, padding, dilation)
    return out[sample].cpu().double(), ref, mag, c * r * s


def _workspace_bytes(name, dtype):
    n, c, h, w, k, r, s, stride, padding, dilation = CASES[name]
    a = _C.Conv2dArgs()
    a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = n, c, h, w, k, r, s
    (a.stride_h, a.stride_w), (a.pad_h, a.pad_w), (a.dil_h, a.dil_w) = stride, padding, dilation
    a.dtype, a.out_f32 = dtype, dtype == _C.F32
    return _C.load().tnx_conv2d_workspace_bytes(ctypes.byref(a))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_packed_conv2d(name, dtype, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    code = {torch.bfloat16: _C.BF16, torch.float16: _C.F16, torch.float32: _C.F32}[dtype]
    assert _workspace_bytes(name, code) > 0
    out, ref, mag, k = _run(name, dtype, device)
    unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dtype]
    per_product = 2.0 ** -16 if dtype == torch.float32 else 0.0
    bound = unit * ref.abs() + (k * 2.0 ** -24 + per_product) * mag + 1e-7
    assert bool(((out - ref).abs() <= bound).all()), ((out - ref).abs() / bound).max().item()


def test_a_non_finite_input_reaches_only_its_own_window(device, monkeypatch):
    """Padded channels and the slabs' padding past k multiply zeros of the scratch, never other pixels."""
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 20, 9, 9, generator=g).bfloat16()
    wt = torch.rand(16, 20, 3, 3, generator=g).add(0.5).bfloat16()
    x[1, 19, 4, 4] = float("inf")
    out = conv2d_forward(x.to(device), wt.to(device), None, (1, 1), (1, 1)).cpu()
    hit = torch.zeros(2, 16, 9, 9, dtype=torch.bool)
    hit[1, :, 3:6, 3:6] = True
    assert bool(torch.isposinf(out[hit]).all()) and bool(torch.isfinite(out[~hit]).all())


@pytest.mark.parametrize("c_in", [32, 33, 64])
def test_non_finite_float32_elements(c_in, device, monkeypatch):
    """Infinities and NaN of either operand fall where the float32 convolution has them, against partners whose bf16 tail is
    zero or of the other sign, zeros, and each other."""
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    g = torch.Generator().manual_seed(c_in)
    inf, nan = float("inf"), float("nan")
    x, wt = torch.randn(2, c_in, 8, 9, generator=g), torch.randn(20, c_in, 3, 3, generator=g)
    x[:, :16], wt[:, :16] = x[:, :16].bfloat16().float(), wt[:, :16].bfloat16().float()
    x[0, 3, 2, 2], x[0, c_in - 1, 6, 6], x[1, 5, 4, 4], x[1, 9, 0, 8] = inf, -inf, nan, inf
    wt[4, 9, 1, 1], wt[7, 3, 0, 2], wt[11, c_in - 1, 2, 2], wt[13, 2, 1, 0] = inf, 0.0, -inf, nan
    out = conv2d_forward(x.to(device), wt.to(device), None, (1, 1), (1, 1)).cpu()
    # the float64 convolution pads with zeros that meet wt's infinities as well: so does every implementation
    ref = torch.nn.functional.conv2d(x.double(), wt.double(), None, 1, 1)
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isnan(out), torch.isnan(ref)) and torch.equal(torch.isposinf(out), torch.isposinf(ref))
    assert torch.equal(torch.isneginf(out), torch.isneginf(ref))
    assert ((out[fin] - ref[fin]).abs().max() / ref[fin].abs().max()).item() < 1e-4
