"""A column-major left operand (`x.t() @ dy`) on the DMA kernels that read it with transposing LDS loads: the same products
in the same order as on the row-major copy of the operand, so the results agree bit for bit."""
import importlib

import pytest
import torch

import tritonix_amd
from tritonix_amd import _C

mm = importlib.import_module("tritonix_amd.ops.matmul")
sg = importlib.import_module("tritonix_amd.ops.swiglu")
pytestmark = pytest.mark.gpu
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8}


def _tiles():
    out = []
    for name in _C.kernel_names():
        f = name.split()
        if "at" in f[6:]:
            out.append((f[0], *(int(v) for v in f[1:6])))
    return out


def _matrix(rows, cols, dtype, gen, device, pad=0, offset=0):
    """[rows, cols] with row pitch cols + pad inside a buffer whose other elements are NaN (int8: 77)."""
    buf = torch.full((rows * (cols + pad) + 64,), 77 if dtype == torch.int8 else float("nan"), dtype=dtype)
    mat = buf[offset:offset + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
    mat.copy_(torch.randint(-127, 128, (rows, cols), generator=gen).to(dtype) if dtype == torch.int8 else torch.randn(rows, cols, generator=gen).to(dtype))
    return buf.to(device)[offset:offset + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]


@pytest.mark.parametrize("tile", _tiles(), ids=lambda t: "-".join(map(str, t)))
def test_transposed_a_matches_the_row_major_kernel(tile, device):
    dt, bm, bn, bk, nw, st = tile
    dtype = DTYPES[dt]
    gen = torch.Generator().manual_seed(bm + bn)
    # whole tiles; ragged in every dimension off 16 bytes; one slab and less; m of one chunk
    for m, n, k, pad, off in ((2 * bm, bn, 4 * bk, 0, 0), (bm + 5, 2 * bn - 3, 3 * bk + 7, 3, 1), (33, 70, bk - 24, 0, 0), (16, 24, bk, 1, 5)):
        a = _matrix(k, m, dtype, gen, device, pad, off).t()
        b = _matrix(k, n, dtype, gen, device, pad, off)
        for split in (1, 2):
            cfg = dict(block_m=bm, block_n=bn, block_k=bk, group_m=8, num_stages=st, num_warps=nw, split_k=split)
            got = mm._launch_matmul(a, b, cfg)
            want = mm._launch_matmul(a.contiguous(), b, cfg)
            assert torch.equal(got, want), (tile, m, n, k, pad, off, split)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.int8], ids=["bf16", "f16", "i8"])
@pytest.mark.parametrize("m,n,k", [(512, 384, 256), (48, 4096, 2048), (1025, 130, 77), (3072, 3072, 192), (2, 1024, 256), (1, 64, 1000)])
def test_wrappers_take_a_transposed_a_as_it_is(m, n, k, dtype, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    gen = torch.Generator().manual_seed(m)
    x, dy = _matrix(k, m, dtype, gen, device), _matrix(k, n, dtype, gen, device)
    got = tritonix_amd.triton_matmul(x.t(), dy)
    if dtype == torch.int8:
        assert torch.equal(got.cpu(), (x.cpu().t().double() @ dy.cpu().double()).to(torch.int32))
        return
    ref = x.cpu().t().double() @ dy.cpu().double()
    mag = x.cpu().t().double().abs() @ dy.cpu().double().abs()
    # exact products, fp32 sums (k * 2^-24 of the magnitudes), one rounding of the result (half a unit: 2^-9 / 2^-12)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert bool(((got.cpu().double() - ref).abs() <= unit * ref.abs() + k * 2.0 ** -24 * mag + 1e-7).all())
    if n % 2 == 0:
        assert torch.equal(sg.glu(x.t(), dy), sg.glu(x.t().contiguous(), dy))
