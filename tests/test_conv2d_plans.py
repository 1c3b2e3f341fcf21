"""The plans of conv2d's packed and window routes that a thread keeps by the layer's sizes: every layer of a program keeps its own, and a
kept plan is the one that a thread that has met nothing makes."""
import ctypes
import random
import threading
import time

from tritonix_amd import _C


def _layers(count, seed):
    rng, out, seen = random.Random(seed), [], set()
    while len(out) < count:
        f, batch, c, k, hw = rng.choice([2, 3, 3, 5]), rng.choice([1, 8, 32]), rng.randrange(32, 257, 32), rng.randrange(32, 513, 8), rng.choice([8, 14, 16, 28, 32, 48, 56])
        stride, dtype = rng.choice([1, 1, 2]), rng.choice([_C.BF16, _C.F16, _C.F32])
        if (f, batch, c, k, hw, stride, dtype) in seen:
            continue
        seen.add((f, batch, c, k, hw, stride, dtype))
        a = _C.Conv2dArgs()
        a.batch, a.c_in, a.h_in, a.w_in, a.c_out, a.filter_h, a.filter_w = batch, c, hw, hw, k, f, f
        a.stride_h = a.stride_w = stride
        a.pad_h = a.pad_w = f // 2
        a.dil_h = a.dil_w = 1
        a.dtype, a.out_f32 = dtype, dtype == _C.F32
        out.append(a)
    return out


def _plan(a):
    info, tile = (ctypes.c_int32 * 6)(), (ctypes.c_int32 * 3)()
    lib = _C.load()
    need, again = lib.tnx_conv2d_workspace_bytes(ctypes.byref(a)), lib.tnx_conv2d_packed_info(ctypes.byref(a), -1, 1, info)
    given = _C.Conv2dArgs.from_buffer_copy(a)
    given.workspace = 4096                       # never dereferenced
    return need, again, tuple(info), lib.tnx_conv2d_route(ctypes.byref(given), tile), tuple(tile)


def _in_a_new_thread(fn):
    got = []
    t = threading.Thread(target=lambda: got.append(fn()))
    t.start()
    t.join()
    return got[0]


def _seconds(layers):
    fn, refs = _C.load().tnx_conv2d_workspace_bytes, [ctypes.byref(a) for a in layers]
    start = time.perf_counter()
    for a in refs:
        fn(a)
    return (time.perf_counter() - start) / len(refs)


def test_every_layer_of_a_network_keeps_its_plan():
    """Finding a plan is a tenth of making one; with layers that push one another out it came to two thirds."""
    layers = _layers(120, 1)
    met, first = _in_a_new_thread(lambda: (_seconds(layers), min(_seconds(layers) for _ in range(50)))[1]), []
    for _ in range(10):
        first.append(_in_a_new_thread(lambda: _seconds(layers)))
    assert met < 0.4 * min(first), (met, min(first))


def test_kept_plans_are_the_ones_made_first():
    layers = _layers(700, 2)                     # more than are kept, on both routes
    routes = [_plan(a)[3] for a in layers]
    assert min(routes.count(_C.CONV_ROUTE_PACKED), routes.count(_C.CONV_ROUTE_WINDOW)) >= 50          # (66 of the drawn ones)
    rng = random.Random(3)
    for rounds in range(3):
        order = list(range(len(layers)))
        rng.shuffle(order)
        for i in order[:250]:                    # one layer, again, and one whose sizes differ in one place
            want = _in_a_new_thread(lambda: _plan(layers[i])) if rounds == 0 and i < 40 else None
            got = _plan(layers[i])
            assert got == _plan(layers[i]) and want in (None, got)
            a = _C.Conv2dArgs.from_buffer_copy(layers[i])
            a.c_out += 1
            other = _plan(a)
            a.c_out -= 1
            assert _plan(a) == got, (i, other)
    assert [_plan(a) for a in layers] == _in_a_new_thread(lambda: [_plan(a) for a in reversed(layers)])[::-1]


def test_what_a_bias_or_a_tile_changes():
    a = _layers(1, 4)[0]
    a.dtype, a.out_f32 = _C.BF16, 0
    taken = _plan(a)
    assert taken[0] > 0
    a.bias, a.bias_dtype = 4096, 17              # never dereferenced: a type that there is not
    assert _plan(a)[0] == 0
    for dtype in (_C.F16, _C.BF16, _C.F32):
        a.bias_dtype = dtype
        assert _plan(a) == taken == _in_a_new_thread(lambda: _plan(a))
    a.bias = None
    a.block_cout, a.block_pixels, a.block_k = 128, 64, 64
    assert _plan(a)[0] == 0
    a.block_cout = a.block_pixels = a.block_k = 0
    a.loader = _C.CONV_LOADER_REGISTERS
    assert _plan(a)[0] == 0
    a.loader = _C.CONV_LOADER_AUTO
    assert _plan(a) == taken
