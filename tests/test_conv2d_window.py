"""conv2d on tiles that keep their input window in LDS (conv_halo.h): the window's size on the CPU, every tile at ragged edges.

Bound: products of 16-bit operands are exact in fp32 and summed in fp32, at most k * 2^-24 of the sum of magnitudes off before the one
rounding, which is half a unit of 2^-8 (bf16) or 2^-11 (f16)."""
import ctypes
import random

import pytest
import torch

from tritonix_amd import _C
from tritonix_amd.ops.conv2d import conv2d_forward

CODES = {torch.bfloat16: _C.BF16, torch.float16: _C.F16, torch.float32: _C.F32}
FIRST, TILES = 64, 16
# n, c_in, h, w, c_out, r, s, stride, padding, dilation
LAYERS = {
    "whole_blocks": (3, 64, 13, 11, 277, 3, 3, (1, 1), (1, 1), (1, 1)),
    "ragged_channels": (2, 117, 16, 24, 70, 3, 3, (1, 1), (1, 1), (1, 1)),
    "one_block": (3, 17, 12, 10, 5, 3, 3, (1, 1), (1, 1), (1, 1)),
    "stride_2": (2, 72, 27, 23, 130, 3, 3, (2, 2), (1, 1), (1, 1)),
    "stride_2_even_padding": (2, 40, 17, 18, 33, 5, 5, (2, 2), (2, 2), (1, 1)),
    "stride_3_dilated": (2, 40, 23, 19, 64, 2, 3, (3, 2), (2, 3), (2, 2)),
    "images_below_a_tile": (9, 64, 7, 7, 200, 3, 3, (1, 1), (1, 1), (1, 1)),
    "pad_wider_than_image": (1, 33, 3, 2, 24, 5, 5, (1, 1), (4, 4), (1, 1)),
    "one_output": (1, 64, 5, 5, 33, 5, 5, (1, 1), (0, 0), (1, 1)),
    "2x2": (2, 96, 20, 20, 64, 2, 2, (1, 1), (0, 0), (1, 1)),
    "whole_rows": (2, 96, 28, 28, 128, 3, 3, (1, 1), (1, 1), (1, 1)),
}


def _args(layer, dtype):
    n, c, h, w, k, r, s, stride, padding, dilation = layer
    a = _C.Conv2dArgs()
    a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = n, c, h, w, k, r, s
    (a.stride_h, a.stride_w), (a.pad_h, a.pad_w), (a.dil_h, a.dil_w) = stride, padding, dilation
    a.dtype, a.out_f32 = CODES[dtype], dtype == torch.float32
    return a


def _info(a, tile, narrower=0):
    info = (ctypes.c_int32 * 6)()
    return _C.load().tnx_conv2d_packed_info(ctypes.byref(a), tile, narrower + 1, info), tuple(info)


def test_window_rows_hold_every_tap_of_every_tile():
    rng = random.Random(5)
    for _ in range(300):
        stride, dil = (rng.choice([1, 1, 2, 3]), rng.choice([1, 1, 2])), (rng.choice([1, 1, 2, 3]), rng.choice([1, 2]))
        layer = (rng.choice([1, 2, 3, 5]), rng.choice([8, 40, 64]), rng.randint(1, 30), rng.randint(1, 30), 40, rng.choice([2, 3, 5]), rng.choice([2, 3, 5]),
                 stride, (rng.randint(0, 4), rng.randint(0, 4)), dil)
        a = _args(layer, torch.bfloat16)
        h_out, w_out = ctypes.c_int32(), ctypes.c_int32()
        _C.load().tnx_conv2d_output_size(ctypes.byref(a), ctypes.byref(h_out), ctypes.byref(w_out))
        h_out, w_out = h_out.value, w_out.value
        tile, narrower = FIRST + rng.randrange(TILES), rng.choice([0, 0, 1, 2, 5])
        if h_out <= 0 or w_out <= 0 or not _info(a, tile, narrower)[0]:
            continue
        _, (_, bn, _, _, rows, lds) = _info(a, tile, narrower)
        width, span = bn - 8 * narrower, (layer[5] - 1) * dil[0] + 1
        hwp, image = -(-h_out * w_out // 8) * 8, (h_out - 1) * stride[0] + span

        def row(pixel):
            r = min(pixel % hwp, h_out * w_out - 1)
            return pixel // hwp * image + r // w_out * stride[0]

        total = layer[0] * hwp
        most = max(row(min(p + width, total) - 1) - row(p) + span for p in range(0, total, width))
        assert most <= rows and lds <= 163840, (layer, tile, narrower, most, rows)


def test_places_behind_the_table_of_taps_are_whole_chunks():
    """The 16-byte places that end a workgroup's LDS follow windows of whole slots and a table of 4 bytes per k step."""
    seen = set()
    for tile in range(FIRST, FIRST + TILES):
        for c in range(8, 400, 8):
            need, info = _info(_args((2, c, 12, 10, 64, 3, 3, (1, 1), (1, 1), (1, 1)), torch.bfloat16), tile)
            if need:
                assert info[5] % 16 == 0, (tile, c, info)
                seen.add(tile)
    assert len(seen) == TILES


def _route(layer, dtype, workspace=True):
    a, tile = _args(layer, dtype), (ctypes.c_int32 * 3)()
    a.workspace = 4096 if workspace else None               # never dereferenced
    return _C.load().tnx_conv2d_route(ctypes.byref(a), tile), tuple(tile)


def test_which_route_a_call_takes():
    bf16, unit = torch.bfloat16, ((1, 1), (1, 1), (1, 1))
    # layers that the margins leave to the windows by far, and tiles that were built for them
    for layer in ((32, 256, 56, 56, 256, 3, 3) + unit, (32, 128, 56, 56, 128, 3, 3, (2, 2), (1, 1), (1, 1)), (32, 128, 28, 28, 128, 3, 3) + unit,
                  (128, 64, 28, 28, 64, 3, 3) + unit):
        for dtype in (bf16, torch.float16):
            route, (bm, width, cut) = _route(layer, dtype)
            tiles = [info for info in (_info(_args(layer, dtype), t)[1] for t in range(FIRST, FIRST + TILES)) if info[0] == bm and info[1] >= width]
            assert route == _C.CONV_ROUTE_WINDOW and width % 8 == 0 and tiles and cut == 1
        assert _route(layer, torch.float32)[0] == _C.CONV_ROUTE_PACKED
        assert _route(layer, bf16, workspace=False)[0] in (_C.CONV_ROUTE_DMA, _C.CONV_ROUTE_REGISTERS)
    # one row or column of taps, channels that are a fifth padding, few outputs
    for layer in ((32, 128, 28, 28, 128, 1, 3) + unit, (32, 128, 28, 28, 128, 3, 1) + unit, (32, 40, 56, 56, 128, 3, 3) + unit, (1, 512, 7, 7, 512, 3, 3) + unit,
                  (32, 256, 56, 56, 256, 1, 1, (2, 2), (0, 0), (1, 1))):
        assert _route(layer, bf16)[0] == _C.CONV_ROUTE_PACKED, layer
    assert _route((32, 256, 56, 56, 256, 1, 1, (1, 1), (0, 0), (1, 1)), bf16)[0] == _C.CONV_ROUTE_GEMM
    assert _route((1, 8, 2, 2, 8, 5, 5, (1, 1), (0, 0), (1, 1)), bf16) == (0, (0, 0, 0))


def test_what_the_tiles_do_not_take():
    ok = LAYERS["whole_blocks"]
    assert _info(_args(ok, torch.bfloat16), FIRST)[0] > 0 and _info(_args(ok, torch.float16), FIRST + TILES - 1)[0] > 0
    assert _info(_args(ok, torch.bfloat16), FIRST + TILES)[0] == 0 and _info(_args(ok, torch.float32), FIRST)[0] == 0
    assert _info(_args(ok, torch.bfloat16), FIRST, 300)[0] == 0                                           # no pixel left
    for r, s, stride in ((1, 3, (1, 1)), (3, 1, (1, 1)), (3, 3, (1, 3))):
        assert _info(_args(ok[:5] + (r, s, stride) + ok[8:], torch.bfloat16), FIRST)[0] == 0
    assert _info(_args((1, 64, 200, 400, 64, 3, 3, (2, 2), (1, 1), (1, 1)), torch.bfloat16), FIRST)[0] == 0    # windows past the LDS
    # the workspace is the packed route's, whichever is taken
    a = _args((64, 256, 56, 56, 64, 3, 3, (1, 1), (1, 1), (1, 1)), torch.bfloat16)
    assert _C.load().tnx_conv2d_workspace_bytes(ctypes.byref(a)) == _info(a, -1)[0] > 100 << 20


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
            unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
            made[name, dtype] = (x.to(device), wt.to(device), b.to(device), ref, unit * ref.abs() + c * r * s * 2.0 ** -24 * mag + 1e-7)
        return made[name, dtype]

    return get


def _bind(a, x, w, b, out, ws):
    a.input, a.weight, a.bias, a.output = x.data_ptr(), w.data_ptr(), b.data_ptr() if b is not None else None, out.data_ptr()
    a.bias_dtype, a.workspace, a.workspace_bytes = CODES[b.dtype] if b is not None else 0, ws.data_ptr(), ws.numel()
    a.out_f32 = out.dtype == torch.float32
    a.stream = torch.cuda.current_stream().cuda_stream


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("tile", range(FIRST, FIRST + TILES))
def test_every_window_tile(tile, dtype, device, problems):
    lib, ran = _C.load(), 0
    for name, layer in LAYERS.items():
        x, w, b, ref, bound = problems(name, dtype, device)
        for narrower in (0, 2):
            a = _args(layer, dtype)
            need, _ = _info(a, tile, narrower)
            if not need:
                continue
            ran += 1
            if narrower:                                    # from an odd element on, infinities around the tensor
                around = torch.full((x.numel() + 64,), float("inf"), dtype=dtype, device=device)
                x = around[33:33 + x.numel()].view(x.shape).copy_(x)
            out = torch.full(ref.shape, float("nan"), dtype=dtype, device=device)
            _bind(a, x, w, b, out, torch.empty(need, dtype=torch.uint8, device=device).fill_(255))
            assert lib.tnx_conv2d_packed_forward(ctypes.byref(a), tile, narrower + 1) == _C.OK
            worst = ((out.cpu().double() - ref).abs() / bound).max().item()
            assert worst <= 1.0, (name, narrower, worst)
    assert ran >= 10


@pytest.mark.gpu
def test_binary32_output_and_bias(device, problems):
    x, w, b, _, _ = problems("ragged_channels", torch.bfloat16, device)
    layer = LAYERS["ragged_channels"]
    ref = torch.nn.functional.conv2d(x.double().cpu(), w.double().cpu(), b.double().cpu(), *layer[7:])
    for bias, want in ((b.float(), ref), (None, ref - b.double().cpu()[None, :, None, None])):
        a = _args(layer, torch.bfloat16)
        out = torch.full(ref.shape, float("nan"), device=device)
        _bind(a, x, w, bias, out, torch.empty(_info(a, FIRST + 4)[0], dtype=torch.uint8, device=device))
        assert _C.load().tnx_conv2d_packed_forward(ctypes.byref(a), FIRST + 4, 1) == _C.OK
        # 1,053 products of unit variance each times 1/1053: sums of magnitudes stay below 40
        assert (out.cpu().double() - want).abs().max().item() <= 1053 * 2.0 ** -24 * 40


@pytest.mark.gpu
def test_the_route_is_taken_by_the_call_and_replays(device, monkeypatch):
    """A layer the library's choice gives to the window tiles, through the public call, in a graph with new operands for each replay: the bits
    are those of a window tile (any of them sums in the same order), which are not the packed route's."""
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    layer = (32, 128, 28, 28, 128, 3, 3, (1, 1), (1, 1), (1, 1))
    route, (bm, _, _) = _route(layer, torch.bfloat16)
    assert route == _C.CONV_ROUTE_WINDOW

    def forced(tile):
        a, out = _args(layer, torch.bfloat16), torch.empty(32, 128, 28, 28, dtype=torch.bfloat16, device=device)
        need, info = _info(a, tile)
        _bind(a, x, w, None, out, torch.empty(need, dtype=torch.uint8, device=device))
        assert _C.load().tnx_conv2d_packed_forward(ctypes.byref(a), tile, 1) == _C.OK
        return out, info

    x, w = torch.randn(32, 128, 28, 28, device=device).bfloat16(), (torch.randn(128, 128, 3, 3, device=device) / 34).bfloat16()
    args = (x, w, None, (1, 1), (1, 1), (1, 1))
    conv2d_forward(*args)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = conv2d_forward(*args)
    for seed in range(4):
        x.normal_(generator=torch.Generator(device).manual_seed(seed))
        w.normal_(0.0, 1 / 34, generator=torch.Generator(device).manual_seed(seed + 9))
        graph.replay()
        eager = conv2d_forward(*args)
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        window, info = forced(next(t for t in range(FIRST, FIRST + TILES) if _info(_args(layer, torch.bfloat16), t)[1][0] == bm))
        assert info[0] == bm and torch.equal(out, window) and not torch.equal(out, forced(-1)[0])
        ref = torch.nn.functional.conv2d(x[:2].cpu().double(), w.cpu().double(), None, 1, 1)
        assert ((out[:2].cpu().double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1152 * 2.0 ** -24 * 40).all()


@pytest.mark.gpu
def test_a_non_finite_input_reaches_only_its_own_window(device):
    """Padded channels, and what an unaligned row piece brings along of its neighbour, never meet another pixel."""
    g = torch.Generator().manual_seed(3)
    layer = (2, 52, 9, 9, 16, 3, 3, (1, 1), (1, 1), (1, 1))
    x, w = torch.randn(2, 52, 9, 9, generator=g).bfloat16(), torch.rand(16, 52, 3, 3, generator=g).add(0.5).bfloat16()
    x[1, 51, 4, 0], x[0, 0, 8, 8] = float("inf"), float("inf")
    hit = torch.zeros(2, 16, 9, 9, dtype=torch.bool)
    hit[1, :, 3:6, 0:2] = True
    hit[0, :, 7:9, 7:9] = True
    xd, wd = x.to(device), w.to(device)
    for tile in range(FIRST, FIRST + TILES):
        a = _args(layer, torch.bfloat16)
        need, _ = _info(a, tile)
        if need:
            out = torch.empty(2, 16, 9, 9, dtype=torch.bfloat16, device=device)
            _bind(a, xd, wd, None, out, torch.empty(need, dtype=torch.uint8, device=device).fill_(255))
            assert _C.load().tnx_conv2d_packed_forward(ctypes.byref(a), tile, 1) == _C.OK
            got = out.cpu()
            assert bool(torch.isposinf(got[hit]).all()) and bool(torch.isfinite(got[~hit]).all()), tile
