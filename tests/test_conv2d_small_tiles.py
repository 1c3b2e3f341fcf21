"""The packed conv2d tiles of 32 channels and of two ring slots, uncut and cut along K, at ragged edges (bounds as in
test_gpu_conv2d_packed.py), and the choice of the route for layers of few multiply-adds per output."""
import ctypes

import pytest
import torch

from test_conv2d_packed_tiles import CODES, LAYERS, _args, _info, problems  # noqa: F401  (a fixture)
from tritonix_amd import _C

FIRST = 32
TILES = [(32, 64, 4, 4), (32, 128, 4, 3), (32, 128, 4, 2), (32, 256, 4, 2), (64, 64, 4, 2), (64, 128, 8, 2)]


def test_the_table_holds_these_tiles_too():
    for dtype in CODES:
        a = _args(LAYERS["whole_slabs"], dtype)
        for i, tile in enumerate(TILES):
            nbytes, info = _info(a, FIRST + i, 3)
            assert nbytes > 0 and info == tile + (3, 2 if dtype == torch.float32 else 1)
        assert _info(a, FIRST + len(TILES), 1)[0] == 0 and _info(a, FIRST - 1, 1)[0] == 0


@pytest.mark.parametrize("layer, packed", [
    ((1, 3, 17, 17, 45, 3, 3, (1, 1), (1, 1), (1, 1)), False), ((64, 3, 112, 112, 64, 3, 3, (1, 1), (1, 1), (1, 1)), True),
    ((64, 3, 7, 7, 32, 3, 3, (1, 1), (1, 1), (1, 1)), False), ((128, 36, 56, 56, 960, 1, 1, (2, 2), (0, 0), (1, 1)), True),
    ((32, 64, 14, 14, 27, 1, 1, (2, 2), (0, 0), (1, 1)), False), ((1, 17, 9, 9, 8, 3, 3, (1, 1), (1, 1), (1, 1)), True)])
def test_few_multiply_adds_take_the_route_that_is_faster(layer, packed):
    for dtype in (torch.bfloat16, torch.float16):
        assert (_info(_args(layer, dtype))[0] > 0) == packed
    assert _info(_args(layer, torch.float32))[0] > 0            # its alternative is three launches


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(CODES), ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("tile", range(len(TILES)), ids=["x".join(map(str, t[:2])) + f"w{t[2]}s{t[3]}" for t in TILES])
def test_every_small_tile(tile, dtype, device, problems):  # noqa: F811
    lib = _C.load()
    for name, layer in LAYERS.items():
        x, w, b, ref, bound = problems(name, dtype, device)
        for split in (1, 3, 16):
            a = _args(layer, dtype)
            need, _ = _info(a, FIRST + tile, split)
            out = torch.full(ref.shape, float("nan"), dtype=dtype, device=device)
            ws = torch.empty(need, dtype=torch.uint8, device=device)
            a.input, a.weight, a.bias, a.output = x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr()
            a.bias_dtype, a.workspace, a.workspace_bytes = CODES[dtype], ws.data_ptr(), need
            a.stream = torch.cuda.current_stream().cuda_stream
            assert lib.tnx_conv2d_packed_forward(ctypes.byref(a), FIRST + tile, split) == _C.OK
            worst = ((out.cpu().double() - ref).abs() / bound).max().item()
            assert worst <= 1.0, (name, split, worst)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(CODES), ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("layer", [(8, 3, 64, 64, 97, 3, 3, (1, 1), (1, 1), (1, 1)), (40, 11, 31, 29, 200, 3, 3, (2, 1), (1, 2), (1, 1)),
                                   (16, 36, 57, 55, 515, 1, 1, (2, 2), (0, 0), (1, 1)), (2, 3, 40, 40, 33, 3, 3, (1, 1), (4, 4), (4, 4)),
                                   (4, 19, 17, 17, 300, 1, 1, (1, 1), (0, 0), (1, 1))])
def test_few_multiply_adds(layer, dtype, device, monkeypatch):
    """The layers whose route is priced, through the public call, against a float64 convolution."""
    from tritonix.ops.conv2d import conv2d_forward

    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    n, c, h, w, k, r, s, stride, padding, dilation = layer
    g = torch.Generator().manual_seed(n + c)
    x, wt = torch.randn(n, c, h, w, generator=g).to(dtype), (torch.randn(k, c, r, s, generator=g) / (c * r * s) ** 0.5).to(dtype)
    b = torch.randn(k, generator=g).to(dtype)
    ref = torch.nn.functional.conv2d(x.double(), wt.double(), b.double(), stride, padding, dilation)
    mag = torch.nn.functional.conv2d(x.double().abs(), wt.double().abs(), b.double().abs(), stride, padding, dilation)
    unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dtype]
    bound = unit * ref.abs() + (c * r * s * 2.0 ** -24 + (2.0 ** -16 if dtype == torch.float32 else 0.0)) * mag + 1e-7
    out = conv2d_forward(x.to(device), wt.to(device), b.to(device), stride, padding, dilation)
    assert ((out.cpu().double() - ref).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("layer", [(3, 200, 14, 14, 30), (2, 64, 33, 33, 640), (5, 23, 17, 17, 70), (1, 130, 7, 7, 129), (16, 3, 33, 33, 515),
                                   (9, 1000, 9, 11, 61)])
def test_images_of_a_1x1_layer(layer, dtype, device, monkeypatch):
    """1x1 layers on every kind of tile the choice gives them: channels, pixels and planes that end inside a tile."""
    from tritonix.ops.conv2d import conv2d_forward

    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    n, c, h, w, k = layer
    g = torch.Generator().manual_seed(n + c)
    x, wt, b = torch.randn(n, c, h, w, generator=g).to(dtype), (torch.randn(k, c, 1, 1, generator=g) / c ** 0.5).to(dtype), torch.randn(k, generator=g).to(dtype)
    ref = torch.nn.functional.conv2d(x.double(), wt.double(), b.double())
    mag = torch.nn.functional.conv2d(x.double().abs(), wt.double().abs(), b.double().abs())
    bound = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype] * ref.abs() + c * 2.0 ** -24 * mag + 1e-7
    out = conv2d_forward(x.to(device), wt.to(device), b.to(device))
    assert ((out.cpu().double() - ref).abs() <= bound).all()
