"""Nothing that the direct-to-LDS ring loads lies outside the operands.

The ring moves a k row (a row of a row-major B, or of an m-contiguous A) in whole 16-byte chunks, the last of them too
where the row ends inside it; the slabs that ``tnx_gemm_tail_slabs`` counts go element by element.  So the last k row in the
ring must start at least a chunk's end before the operand does.  Recomputed here from that sentence, no GPU; then the same
sizes against the exact product on one."""
import ctypes
import importlib

import pytest
import torch

from tritonix_amd import _C

mm = importlib.import_module("tritonix_amd.ops.matmul")
TYPES = {"f16": (_C.F16, _C.F16, 2), "bf16": (_C.BF16, _C.BF16, 2), "i8": (_C.I8, _C.I32, 1)}


def _args(dt, tile, m, n, k, a_strides, b_strides, misaligned=0):
    g = _C.GemmArgs()
    g.m, g.n, g.k = m, n, k
    (g.stride_am, g.stride_ak), (g.stride_bk, g.stride_bn), (g.stride_cm, g.stride_cn) = a_strides, b_strides, (n, 1)
    g.in_dtype, g.out_dtype, _ = TYPES[dt]
    g.block_m, g.block_n, g.block_k, g.num_warps, g.num_stages = tile
    g.group_m, g.split_k = 8, 1
    g.a = g.b = 4096 + misaligned                     # never dereferenced: the alignment counts
    return g


def _inside(tail, bk, k, length, pitch, vec):
    """Whether the chunk that ends the last k row of the ring ends inside an operand of k rows."""
    rows = max(0, (-(-k // bk) - tail) * bk)          # k rows in the ring; what is left out includes the partial slab
    return rows == 0 or (rows - 1) * pitch + -(-length // vec) * vec <= (k - 1) * pitch + length


def test_every_tile_on_narrow_operands():
    lib = _C.load()
    checked = elementwise = 0
    for name in _C.kernel_names():
        parts = name.split()
        dt, tile = parts[0], tuple(int(v) for v in parts[1:6])
        bk, vec = tile[2], 16 // TYPES[dt][2]
        for layout in ["nn"] + (["tn"] if "at" in parts else []):
            for k in (1, 3, bk, bk + 1, bk + 2, 2 * bk + 5, 3 * bk - 1, 3 * bk + 1):
                for width in range(1, 2 * vec + 2):
                    for extra in (0, 1):
                        m, n = (width, 40) if layout == "tn" else (40, width)
                        if layout == "tn" and m + extra == 1:
                            continue                  # unit pitch: one row, not this layout
                        g = _args(dt, tile, m, n, k, (1, m + extra) if layout == "tn" else (k, 1), (n + extra, 1))
                        tail = lib.tnx_gemm_tail_slabs(ctypes.byref(g))
                        assert tail >= 0, (name, layout, m, n, k)          # refused nowhere
                        if layout == "tn" or not (n == 1 and extra == 0 and "bt" in parts):      # [k, 1]: also k-contiguous
                            assert _inside(tail, bk, k, n, n + extra, vec), (name, layout, m, n, k, extra, tail)
                        if layout == "tn":
                            assert _inside(tail, bk, k, m, m + extra, vec), (name, layout, m, n, k, extra, tail)
                        elementwise += tail > 1
                        checked += 1
    assert checked > 10000 and elementwise > 100


def test_the_ring_is_left_only_where_it_has_to_be():
    lib = _C.load()
    tile = (64, 64, 64, 4, 4)
    for n, k, want in ((64, 256, 0), (60, 256, 1), (60, 257, 1), (4, 257, 1), (3, 257, 5), (3, 258, 1), (2, 258, 5), (2, 259, 1)):
        assert lib.tnx_gemm_tail_slabs(ctypes.byref(_args("bf16", tile, 64, n, k, (k, 1), (n, 1)))) == want, (n, k)
    assert lib.tnx_gemm_tail_slabs(ctypes.byref(_args("bf16", tile, 64, 64, 256, (256, 1), (64, 1), misaligned=2))) == 1


def _signs(shape, dtype, gen):
    return torch.randint(-1, 2, shape, generator=gen).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.int8])
def test_wrappers_keep_narrow_operands_off_the_ring(dtype):
    """The operands as the wrappers hand them over, and the built-in choice for them: no call on the element-wise loader."""
    lib = _C.load()
    dt = "bf16" if dtype == torch.bfloat16 else "i8"
    for width in range(1, 17):
        for k in (65, 66, 129, 130, 257, 385):
            for a, b in ((torch.zeros(k, width, dtype=dtype).t(), torch.zeros(k, 40, dtype=dtype)),
                         (torch.zeros(40, k, dtype=dtype), torch.zeros(k, width, dtype=dtype))):
                m, n = a.shape[0], b.shape[1]
                x, y, _ = mm.engine_operands(a, b)
                assert torch.equal(x, a) and torch.equal(y, b)
                c = mm.default_config(x, y)
                g = _args(dt, (c["block_m"], c["block_n"], c["block_k"], c["num_warps"], c["num_stages"]), m, n, k, x.stride(), y.stride())
                tail = lib.tnx_gemm_tail_slabs(ctypes.byref(g))
                assert 0 <= tail <= 1, (m, n, k, tail)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.int8], ids=["bf16", "i8"])
@pytest.mark.parametrize("layout", ["nn", "tn"])
def test_narrow_operands(layout, dtype, device, monkeypatch):
    """Products of -1, 0, 1: the sums are exact in fp32 and stay below 2^8, so the 16-bit result is exact too."""
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    import tritonix_amd

    named = dict(block_m=128, block_n=128, block_k=128 // dtype.itemsize, group_m=8, num_stages=3, num_warps=8)   # no element-wise loader
    g = torch.Generator().manual_seed(5)
    for width in (1, 2, 3, 4, 7, 8, 9):
        for k in (65, 66, 129, 130, 193, 257, 1025, 2049):
            m, n = (width, 70) if layout == "tn" else (70, width)
            a, b = _signs((m, k), dtype, g), _signs((k, n), dtype, g)
            ref = a.double() @ b.double()
            assert ref.abs().max() < 256
            ad, bd = a.t().contiguous().to(device).t() if layout == "tn" else a.to(device), b.to(device)
            for out in (tritonix_amd.triton_matmul(ad, bd), mm.matmul_splitk(ad, bd), mm._launch_matmul(ad, bd, named)):
                assert torch.equal(out.cpu().double(), ref), (m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("hw", [1, 2, 3])
def test_1x1_layer_of_tiny_planes(hw, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    from tritonix_amd.ops.conv2d import conv2d_forward

    g = torch.Generator().manual_seed(hw)
    for c_in in (65, 66, 129, 193):
        x, w = _signs((3, c_in, 1, hw), torch.float16, g), _signs((40, c_in, 1, 1), torch.float16, g)
        out = conv2d_forward(x.to(device), w.to(device))
        assert torch.equal(out.cpu().double(), torch.nn.functional.conv2d(x.double(), w.double())), c_in
