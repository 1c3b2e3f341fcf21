"""float32 products at the edges of the one-pass split (tnx_gemm_f32): every operand layout, sizes off the 8-element chunks
and the K slabs it pads to, and the tiles whose binary32 epilogue is a kernel of its own.

Bound: the dropped lo * lo term and the rounding of lo are at most 2^-17 + 2^-17 of a product, fp32 sums add
3k * 2^-24; against the float64 product, per element, on the sum of magnitudes."""
import importlib

import pytest
import torch

import tritonix_amd
from tritonix_amd import _C

mm = importlib.import_module("tritonix_amd.ops.matmul")
sg = importlib.import_module("tritonix_amd.ops.swiglu")
pytestmark = pytest.mark.gpu

LARGE = [(256, 256, 2), (192, 256, 2), (256, 192, 2), (192, 192, 3)]


def _operands(m, n, k, layout, device, seed=0):
    g = torch.Generator().manual_seed(seed + m + n + k)
    a, b = torch.randn(m, k, generator=g), torch.randn(k, n, generator=g) / k ** 0.5
    ad = a.t().contiguous().to(device).t() if layout[0] == "t" else a.to(device)
    bd = b.t().contiguous().to(device).t() if layout[1] == "t" else b.to(device)
    ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    return ad, bd, ref, mag


def _check(out, ref, mag, k, what):
    assert out.dtype == torch.float32
    bound = (2.0 ** -16 + 3 * k * 2.0 ** -24) * mag + 1e-30
    assert bool(((out.cpu().double() - ref).abs() <= bound).all()), what


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (17, 33, 9), (64, 100, 64), (129, 257, 65), (300, 40, 1000), (513, 770, 22)])
def test_built_in_choice(m, n, k, layout, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    a, b, ref, mag = _operands(m, n, k, layout, device)
    _check(tritonix_amd.triton_matmul(a, b), ref, mag, k, (m, n, k, layout))


@pytest.mark.parametrize("tile", LARGE, ids=lambda t: "%dx%d" % t[:2])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_large_tiles(tile, layout, device):
    bm, bn, st = tile
    for m, n, k, split in ((2 * bm, bn, 128, 1), (bm + 3, bn + 5, 77, 1), (5, 9, 200, 2), (bm, 2 * bn - 1, 700, 2)):
        a, b, ref, mag = _operands(m, n, k, layout, device)
        cfg = dict(block_m=bm, block_n=bn, block_k=64, group_m=8, num_stages=st, num_warps=8, split_k=split)
        _check(mm._launch_matmul(a, b, cfg), ref, mag, k, (tile, m, n, k, layout, split))


SMALL = [(128, 128, 8, 3), (128, 128, 4, 3), (64, 128, 8, 3), (64, 64, 4, 4)]


@pytest.mark.parametrize("tile", SMALL, ids=lambda t: "%dx%d_w%d" % t[:3])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_blocks_of_heads_and_tails_on_the_smaller_tiles(tile, layout, device):
    """k around one block of 32, fewer slabs than the ring has slots, several trips of the unrolled loop, a K cut."""
    bm, bn, nw, st = tile
    for m, n, k, split in ((bm, bn, 32, 1), (bm + 1, bn + 9, 31, 1), (7, bn - 1, 33, 1), (bm - 3, 2 * bn, 65, 1), (bm, bn + 8, 500, 1),
                           (bm + 5, bn, 257, 2), (33, bn, 900, 4)):
        a, b, ref, mag = _operands(m, n, k, layout, device)
        cfg = dict(block_m=bm, block_n=bn, block_k=64, group_m=8, num_stages=st, num_warps=nw, split_k=split)
        _check(mm._launch_matmul(a, b, cfg), ref, mag, k, (tile, m, n, k, layout, split))


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_non_finite_elements_meet_every_kind_of_partner(layout, device):
    """One non-finite element of a times each kind of element of b and the other way round: infinities of both signs
    against +-inf, NaN, 0, a value bf16 holds exactly (zero tail), one whose tail has the other sign, and the
    smallest normal number.  Infinities and NaN fall where the fp32 product has them."""
    inf, nan = float("inf"), float("nan")
    kinds = [inf, -inf, nan, 0.0, -0.0, 1.0, -1.5, 1.0 + 2.0 ** -9 - 2.0 ** -12, -(1.0 + 2.0 ** -9 - 2.0 ** -12), 1.00390625 + 2.0 ** -10, 2.0 ** -126, -2.0 ** -126]
    a, b = torch.zeros(len(kinds), 40), torch.zeros(40, len(kinds))
    a[:, 35], b[35, :] = torch.tensor(kinds), torch.tensor(kinds)            # one k meets one k: every pair
    a[:, 3], b[3, :] = 2.0, 3.0                                               # and a finite term beside it
    ad = a.t().contiguous().to(device).t() if layout[0] == "t" else a.to(device)
    bd = b.t().contiguous().to(device).t() if layout[1] == "t" else b.to(device)
    cfg = dict(block_m=64, block_n=64, block_k=64, group_m=8, num_stages=4, num_warps=4)
    out, ref = mm._launch_matmul(ad, bd, cfg).cpu(), a @ b
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(torch.isposinf(out), torch.isposinf(ref)) and torch.equal(torch.isneginf(out), torch.isneginf(ref))
    fin = torch.isfinite(ref)
    assert ((out[fin] - ref[fin]).abs() <= 2.0 ** -15 * ref[fin].abs()).all()


def test_gated_product_on_a_large_tile(device):
    g = torch.Generator().manual_seed(4)
    x, w12 = torch.randn(300, 128, generator=g), torch.randn(128, 520, generator=g) / 12
    cfg = dict(block_m=256, block_n=256, block_k=64, group_m=8, num_stages=2, num_warps=8)
    z = sg._launch_glu(x.to(device), w12.to(device), cfg, "silu").cpu()
    y = x.double() @ w12.double()
    ref = torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2]
    assert ((z - ref).abs().max() / ref.abs().max()).item() < 1e-4


def test_scratch_is_checked_before_anything_is_launched(device):
    import ctypes

    lib = _C.load()
    a, b = torch.zeros(64, 64, device=device), torch.zeros(64, 64, device=device)
    c = torch.full((64, 64), 7.0, device=device)
    g = _C.GemmArgs()
    g.a, g.b, g.c, g.m, g.n, g.k = a.data_ptr(), b.data_ptr(), c.data_ptr(), 64, 64, 64
    g.stride_am, g.stride_ak, g.stride_bk, g.stride_bn, g.stride_cm, g.stride_cn = 64, 1, 64, 1, 64, 1
    g.in_dtype = g.out_dtype = _C.F32
    assert lib.tnx_gemm_default_config(ctypes.byref(g)) == _C.OK
    need = lib.tnx_gemm_f32_scratch_bytes(ctypes.byref(g))
    assert need == 2 * 64 * 128 * 2          # heads and tails of two 64 x 64 operands
    scratch = torch.empty(need, dtype=torch.uint8, device=device)
    assert lib.tnx_gemm_f32(ctypes.byref(g), None, need) == _C.E_WORKSPACE
    assert lib.tnx_gemm_f32(ctypes.byref(g), scratch.data_ptr(), need - 1) == _C.E_WORKSPACE
    g.block_m = 96
    assert lib.tnx_gemm_f32(ctypes.byref(g), scratch.data_ptr(), need) == _C.E_UNSUPPORTED
    torch.cuda.synchronize()
    assert bool((c == 7.0).all())
