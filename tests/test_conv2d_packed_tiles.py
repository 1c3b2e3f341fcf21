"""Every tile of the packed conv2d route, uncut and cut along K, plain and on heads and tails, at ragged edges; and which of
them the cases of test_gpu_conv2d_packed.py run on.  Bounds as there."""
import ctypes

import pytest
import torch

from test_gpu_conv2d_packed import CASES
from tritonix_amd import _C

TILES = [(256, 256, 8, 2), (256, 224, 8, 2), (256, 192, 8, 2), (256, 128, 8, 3), (128, 256, 8, 3), (128, 128, 8, 3), (128, 128, 8, 2),
         (64, 256, 8, 3), (64, 128, 8, 3), (64, 128, 4, 3), (64, 64, 4, 4)]
CODES = {torch.bfloat16: _C.BF16, torch.float16: _C.F16, torch.float32: _C.F32}
# n, c_in, h, w, c_out, r, s, stride, padding, dilation: 277 channels and 432 pixel slots are whole tiles of no kind
LAYERS = {"whole_slabs": (3, 128, 13, 11, 277, 3, 3, (1, 1), (1, 1), (1, 1)), "ragged_k": (3, 117, 13, 11, 277, 3, 3, (1, 1), (1, 1), (1, 1)),
          "stride_2": (2, 136, 27, 23, 277, 3, 3, (2, 2), (1, 1), (1, 1)), "one_pixel_more": (1, 129, 17, 17, 65, 3, 3, (1, 1), (1, 1), (1, 1))}


def _args(layer, dtype):
    n, c, h, w, k, r, s, stride, padding, dilation = layer
    a = _C.Conv2dArgs()
    a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = n, c, h, w, k, r, s
    (a.stride_h, a.stride_w), (a.pad_h, a.pad_w), (a.dil_h, a.dil_w) = stride, padding, dilation
    a.dtype, a.out_f32 = CODES[dtype], dtype == torch.float32
    return a


def _info(a, tile=-1, split=1):
    info = (ctypes.c_int32 * 6)()
    nbytes = _C.load().tnx_conv2d_packed_info(ctypes.byref(a), tile, split, info)
    return nbytes, tuple(info)


def test_the_table_holds_these_tiles():
    for dtype in CODES:
        a = _args(LAYERS["whole_slabs"], dtype)
        for i, tile in enumerate(TILES):
            for split in (1, 2, 16):
                nbytes, info = _info(a, i, split)
                assert nbytes > 0 and info == tile + (split, 2 if dtype == torch.float32 else 1)
        assert _info(a, len(TILES), 1)[0] == 0 and _info(a, 0, 17)[0] == 0 and _info(a, 0, 0)[0] == 0
        assert _info(a)[0] == _C.load().tnx_conv2d_workspace_bytes(ctypes.byref(a))


def test_what_the_packed_cases_run_on():
    """K cut where the case is there for it, three terms and heads and tails where the float32 cases say so."""
    for name, layer in CASES.items():
        for dtype in CODES:
            nbytes, info = _info(_args(layer, dtype))
            assert nbytes > 0, (name, dtype)
            if name in ("cut_k", "blocks_cut_k"):
                assert info[4] > 1, (name, dtype, info)
            if name == "many_tiles":
                assert info[:2] == (256, 224) or dtype == torch.float32, info
            if dtype == torch.float32:
                blocks = name in ("one_block", "block_padded", "two_blocks_padded", "blocks_1x1_stride_2", "blocks_cut_k")
                assert not blocks or info[5] == 2, (name, info)
                assert name != "three_terms_33" or info[5] == 3, info
            else:
                assert info[5] == 1


@pytest.fixture(scope="module")
def problems():
    made = {}

    def get(name, dtype, device):
        if (name, dtype) not in made:
            n, c, h, w, k, r, s, stride, padding, dilation = LAYERS[name]
            g = torch.Generator().manual_seed(len(name))
            x, wt = torch.randn(n, c, h, w, generator=g).to(dtype), (torch.randn(k, c, r, s, generator=g) / (c * r * s) ** 0.5).to(dtype)
            b = torch.randn(k, generator=g).to(dtype)
            ref = torch.nn.functional.conv2d(x.double(), wt.double(), b.double(), stride, padding, dilation)
            mag = torch.nn.functional.conv2d(x.double().abs(), wt.double().abs(), b.double().abs(), stride, padding, dilation)
            unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dtype]
            per_product = 2.0 ** -16 if dtype == torch.float32 else 0.0
            bound = unit * ref.abs() + (c * r * s * 2.0 ** -24 + per_product) * mag + 1e-7
            made[name, dtype] = (x.to(device), wt.to(device), b.to(device), ref, bound)
        return made[name, dtype]

    return get


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(CODES), ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("tile", range(len(TILES)), ids=["x".join(map(str, t[:2])) + f"w{t[2]}s{t[3]}" for t in TILES])
def test_every_tile(tile, dtype, device, problems):
    lib = _C.load()
    for name, layer in LAYERS.items():
        x, w, b, ref, bound = problems(name, dtype, device)
        for split in (1, 2, 16):
            a = _args(layer, dtype)
            need, _ = _info(a, tile, split)
            out = torch.full(ref.shape, float("nan"), dtype=dtype, device=device)
            ws = torch.empty(need, dtype=torch.uint8, device=device)
            a.input, a.weight, a.bias, a.output = x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr()
            a.bias_dtype, a.workspace, a.workspace_bytes = CODES[dtype], ws.data_ptr(), need
            a.stream = torch.cuda.current_stream().cuda_stream
            assert lib.tnx_conv2d_packed_forward(ctypes.byref(a), tile, split) == _C.OK
            worst = ((out.cpu().double() - ref).abs() / bound).max().item()
            assert worst <= 1.0, (name, split, worst)
