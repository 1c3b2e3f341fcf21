"""The scratch of the packed conv2d route: asked for only where its size pays, and done without where there is no room."""
import ctypes
import importlib

import pytest
import torch

from tritonix_amd import _C

forward = importlib.import_module("tritonix_amd.ops.conv2d.forward")


def _workspace_bytes(dtype, n, c, h, w, k, f, stride, pad, dil):
    a = _C.Conv2dArgs()
    a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = n, c, h, w, k, f, f
    a.stride_h = a.stride_w = stride
    a.pad_h = a.pad_w = pad
    a.dil_h = a.dil_w = dil
    a.dtype, a.out_f32 = dtype, dtype == _C.F32
    return _C.load().tnx_conv2d_workspace_bytes(ctypes.byref(a))


def test_a_padding_that_dwarfs_the_input_is_not_written_out():
    """Packed images of 10 to 329 times the input cost more than the kernels that pad as they gather (measured: 227 against
    209 us, 415 / 87, 124 / 77, 74 / 43); of 8 to 30 times it where those leave the chip idle, they pay (52 against 895 us)."""
    for dtype in (_C.BF16, _C.F16):
        for layer in ((8, 2048, 33, 33, 256, 3, 1, 36, 36), (128, 512, 7, 7, 64, 3, 1, 60, 60), (32, 256, 14, 14, 256, 5, 1, 72, 36),
                      (128, 64, 17, 17, 256, 3, 1, 60, 60)):
            assert _workspace_bytes(dtype, *layer) == 0, layer
        for layer in ((1, 2048, 33, 33, 256, 5, 1, 72, 36), (4, 512, 5, 5, 16, 5, 1, 6, 3), (8, 2048, 33, 33, 256, 3, 1, 12, 12),
                      (1, 512, 65, 65, 256, 3, 1, 24, 24), (32, 256, 56, 56, 256, 3, 1, 1, 1), (32, 128, 56, 56, 128, 3, 2, 1, 1)):
            assert _workspace_bytes(dtype, *layer) > 0, layer
    assert _workspace_bytes(_C.F32, 128, 512, 7, 7, 64, 3, 1, 24, 24) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("autotune", ["0", "1"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_no_room_for_the_scratch(dtype, autotune, device, monkeypatch):
    """Without scratch the call runs the kernels it had before, tuned or not."""
    monkeypatch.setenv("TRITONIX_AUTOTUNE", autotune)
    g = torch.Generator().manual_seed(2)
    x, w, b = torch.randn(2, 64, 14, 15, generator=g).to(dtype), (torch.randn(40, 64, 3, 3, generator=g) / 24).to(dtype), torch.randn(40, generator=g).to(dtype)
    xd, wd, bd = x.to(device), w.to(device), b.to(device)
    asked = []

    def no_room(nbytes, dev):
        asked.append(nbytes)
        return None

    monkeypatch.setattr(forward, "_scratch", no_room)
    monkeypatch.setattr(forward, "_CONV_FWD_CONFIG_CACHE", {})
    for _ in range(2):
        out = forward.conv2d_forward(xd, wd, bd, (1, 1), (1, 1)).cpu().double()
        ref = torch.nn.functional.conv2d(x.double(), w.double(), b.double(), 1, 1)
        mag = torch.nn.functional.conv2d(x.double().abs(), w.double().abs(), b.double().abs(), 1, 1)
        unit, per_product = (2.0 ** -8, 0.0) if dtype == torch.bfloat16 else (0.0, 2.0 ** -16)
        assert bool(((out - ref).abs() <= unit * ref.abs() + (576 * 2.0 ** -24 + per_product) * mag + 1e-7).all())
    assert asked


@pytest.mark.gpu
def test_scratch_that_does_not_fit_the_device(device):
    assert forward._scratch(1 << 50, device) is None
    assert forward._scratch(1 << 20, device).numel() == 1 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("error", [torch.OutOfMemoryError, ValueError])
def test_a_failing_own_choice_does_not_end_the_search(error, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "1")
    monkeypatch.setattr(forward, "_CONV_FWD_CONFIG_CACHE", {})
    run = forward.Conv2dForwardKernel.run

    def failing(self, *args, **kw):
        if kw["BLOCK_SIZE_M"] == 0:
            raise error("no")
        return run(self, *args, **kw)

    monkeypatch.setattr(forward.Conv2dForwardKernel, "run", failing)
    x, w = torch.randint(-1, 2, (1, 32, 9, 9)).half().to(device), torch.randint(-1, 2, (16, 32, 3, 3)).half().to(device)
    out = forward.conv2d_forward(x, w, None, (1, 1), (1, 1))
    assert torch.equal(out.cpu().double(), torch.nn.functional.conv2d(x.cpu().double(), w.cpu().double(), None, 1, 1))
