"""What a kept launch (tritonix_amd/_launch.so, tritonix_amd/kernel.py) leaves to go wrong around it: buffers of other threads,
numbers of operations, launches that fail, a module that is not there."""
import ctypes
import importlib
import threading
import time
import types
import weakref

import pytest
import torch

import tritonix_amd.kernel as kernel
from tritonix_amd import _C

mm = importlib.import_module("tritonix_amd.ops.matmul")
GEMM = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p)


def test_the_native_side_is_given_the_buffer_itself(monkeypatch):
    """A pointer alone keeps nothing alive while the interpreter lock is given back."""
    buf = torch.zeros(64, dtype=torch.uint8)
    monkeypatch.setattr(kernel, "_workspace", lambda device, stream, nbytes, atomic: buf)
    assert kernel._workspace_of(0, 0, 64, 0) is buf


def test_threads_that_evict_each_others_workspaces(monkeypatch):
    """A buffer may be evicted between its lookup and its move to the end of the list: nobody's call fails for it."""

    class Slow(type(kernel._workspaces)):
        def move_to_end(self, key):
            time.sleep(0.002)
            super().move_to_end(key)

    monkeypatch.setattr(kernel, "_workspaces", Slow())
    monkeypatch.setattr(kernel, "_MAX_WORKSPACES", 1)
    device, errors = torch.device("cpu", 0), []

    def ask(stream):
        try:
            for _ in range(10):
                assert kernel._workspace(device, stream, 64).numel() >= 64
        except Exception as err:                             # noqa: BLE001
            errors.append(err)

    threads = [threading.Thread(target=ask, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


class _Slow(dict):
    """Lets the other threads in between a read and what is made of it."""

    def __len__(self):
        n = super().__len__()
        time.sleep(0.005)
        return n


def test_operations_asked_for_at_once_get_numbers_of_their_own(monkeypatch):
    monkeypatch.setattr(kernel, "_tags", _Slow(matmul=0))
    start, got = threading.Barrier(8), {}

    def ask(i):
        start.wait()
        got[i] = (kernel.plan_tag(("at once", i)), kernel.plan_tag(("at once", 0)))

    threads = [threading.Thread(target=ask, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len({n for n, _ in got.values()}) == 8 and {n for _, n in got.values()} == {got[0][0]}
    assert all(kernel.plan_tag(("at once", i)) == n for i, (n, _) in got.items())


def test_a_number_is_not_given_twice_when_the_tags_are_dropped(monkeypatch):
    monkeypatch.setattr(kernel, "_tags", {"matmul": 0})
    monkeypatch.setattr(kernel, "_plans", kernel._Plans())
    monkeypatch.setattr(kernel, "_MAX_PLANS", 4)
    numbers = [kernel.plan_tag(("dropped", i)) for i in range(12)]
    assert len(set(numbers)) == 12 and 0 not in numbers and kernel.plan_tag("matmul") == 0


def test_a_failed_launch_drops_its_workspace_and_raises(monkeypatch):
    device, buf = torch.device("cuda", 0), torch.zeros(64, dtype=torch.uint8)
    monkeypatch.setattr(kernel, "_workspaces", type(kernel._workspaces)({kernel._workspace_key(device, 7, False): buf, kernel._workspace_key(device, 8, False): buf}))
    g = _C.GemmArgs()
    g.in_dtype, g.split_k = _C.BF16, 4
    with pytest.raises(RuntimeError):
        kernel._launch_failed(0, 7, _C.E_WORKSPACE, bytes(g))
    assert len(kernel._workspaces) == 2                      # refused before anything ran
    with pytest.raises(RuntimeError):
        kernel._launch_failed(0, 7, _C.E_HIP, bytes(g))
    assert list(kernel._workspaces) == [kernel._workspace_key(device, 8, False)]


def _without_module(monkeypatch, how):
    """``kernel`` as in a process in which the module cannot be had."""
    import sys

    import tritonix_amd

    stand_in = None if how == "missing" else types.SimpleNamespace(torch_version="1.0.0")
    monkeypatch.setitem(sys.modules, "tritonix_amd._launch", stand_in)
    if how == "missing":
        monkeypatch.delattr(tritonix_amd, "_launch", raising=False)
    else:
        monkeypatch.setattr(tritonix_amd, "_launch", stand_in, raising=False)
    monkeypatch.setattr(kernel, "_launch", None)
    monkeypatch.setattr(kernel, "_launch_missing", False, raising=False)
    monkeypatch.setattr(kernel, "product", lambda *_: None)


@pytest.mark.parametrize("how", ["missing", "another torch"])
def test_without_the_module_the_ordinary_path_stays(monkeypatch, how):
    _without_module(monkeypatch, how)
    with pytest.warns(RuntimeWarning):
        assert kernel.launch_module() is None
    assert kernel.launch_module() is None and kernel._launch is None          # said once


@pytest.fixture
def kept_split(monkeypatch, device):
    """Operands of a K-split product whose launch is kept, and a way to repeat it with other entry points."""
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    kernel._plans.clear()
    gen = torch.Generator(device).manual_seed(1)
    a, b = torch.randn(16, 4096, generator=gen, device=device).bfloat16(), torch.randn(4096, 256, generator=gen, device=device).bfloat16()
    want = [mm.matmul_splitk(a, b) for _ in range(3)][-1]
    torch.cuda.synchronize()
    hooks = mm.gemm_splitk_kernel.kernel.pre_run_hooks

    def repeat(gemm, workspace=kernel._workspace_of):
        kernel._bind(kernel._launch, gemm, workspace)
        return kernel._launch.product(kernel.plan_tag(("splitk", 4)), a, b, mm._splitk_cfg, hooks)

    yield repeat, want
    kernel._bind(kernel._launch, _C.load().tnx_gemm)


@pytest.mark.gpu
def test_a_replaced_workspace_lives_until_its_launch_is_queued(kept_split, device):
    repeat, want = kept_split
    refs, at_launch = [], []

    def given_away(index, stream, nbytes, atomic):
        buf = torch.zeros(nbytes, dtype=torch.uint8, device=device)      # (nothing else refers to it: replaced by another thread)
        refs.append(weakref.ref(buf))
        return buf

    def launch(p):
        g = _C.GemmArgs.from_address(p)
        buf = refs[-1]()
        at_launch.append(buf is not None and (g.workspace, g.workspace_bytes) == (buf.data_ptr(), buf.numel()))
        return _C.OK

    assert repeat(GEMM(launch), given_away).shape == want.shape and at_launch == [True]
    assert refs[-1]() is None
    assert torch.equal(repeat(_C.load().tnx_gemm), want)


@pytest.mark.gpu
def test_a_launch_that_fails_is_raised_and_not_repeated(kept_split, device):
    repeat, want = kept_split
    key = kernel._workspace_key(device, kernel._stream_of(0), False)
    asked = []

    def launch(p):
        asked.append(_C.GemmArgs.from_address(p).workspace)
        return _C.E_HIP

    buf = kernel._workspaces[key]
    with pytest.raises(RuntimeError):
        repeat(GEMM(launch))
    assert asked == [buf.data_ptr()] and key not in kernel._workspaces
    assert torch.equal(repeat(_C.load().tnx_gemm), want) and kernel._workspaces[key] is not buf


@pytest.mark.gpu
def test_an_interrupt_is_not_swallowed(kept_split, device):
    repeat, want = kept_split

    def raising(error):
        def workspace(*_):
            raise error
        return workspace

    assert repeat(_C.load().tnx_gemm, raising(torch.OutOfMemoryError())) is None          # the ordinary path meets it again
    with pytest.raises(KeyboardInterrupt):
        repeat(_C.load().tnx_gemm, raising(KeyboardInterrupt()))
    assert torch.equal(repeat(_C.load().tnx_gemm), want)


@pytest.mark.gpu
def test_calls_without_the_module(device, monkeypatch):
    _without_module(monkeypatch, "missing")
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    kernel._plans.clear()
    conv = importlib.import_module("tritonix_amd.ops.conv2d.forward")
    monkeypatch.setattr(conv, "_PLANS", {})
    a, b = torch.randn(40, 96, device=device).half(), torch.randn(96, 72, device=device).half()
    x, w = torch.randn(2, 24, 14, 14, device=device).half(), torch.randn(32, 24, 3, 3, device=device).half()
    with pytest.warns(RuntimeWarning):
        products = [mm.triton_matmul(a, b) for _ in range(4)]
        layers = [conv.conv2d_forward(x, w, None, (1, 1), (1, 1), (1, 1)) for _ in range(3)]
    assert all(torch.equal(p, products[0]) for p in products) and all(torch.equal(y, layers[0]) for y in layers)
    assert kernel._launch is None and any(plan for plan in kernel._plans.values())


class _Tagged(torch.Tensor):
    """A subclass like those that carry metadata: results of its methods are of its type."""


@pytest.mark.gpu
def test_a_subclass_keeps_its_type_on_repeated_calls(device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    kernel._plans.clear()
    conv = importlib.import_module("tritonix_amd.ops.conv2d.forward")
    x, w = torch.randn(2, 24, 14, 14, device=device).half(), torch.randn(32, 24, 3, 3, device=device).half()
    want = [conv.conv2d_forward(x, w, None, (1, 1), (1, 1), (1, 1)) for _ in range(3)][-1]
    for _ in range(3):
        y = conv.conv2d_forward(x.as_subclass(_Tagged), w, None, (1, 1), (1, 1), (1, 1))
        assert type(y) is _Tagged and torch.equal(y.as_subclass(torch.Tensor), want)
    assert type(conv.conv2d_forward(x, torch.nn.Parameter(w), None, (1, 1), (1, 1), (1, 1))) is torch.Tensor
    a, b = torch.randn(40, 96, device=device).half(), torch.randn(96, 72, device=device).half()
    want = [mm.triton_matmul(a, b) for _ in range(3)][-1]
    hooks = mm.matmul_kernel.kernel.pre_run_hooks
    assert kernel._launch.product(0, a.as_subclass(_Tagged), b, mm._matmul_cfg, hooks) is None
    assert torch.equal(kernel._launch.product(0, torch.nn.Parameter(a), b, mm._matmul_cfg, hooks), want)


@pytest.mark.gpu
def test_a_kept_conv2d_call_without_room_for_its_scratch(device, monkeypatch):
    """The native side answers None, and the ordinary path runs the kernel that needs none."""
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    conv = importlib.import_module("tritonix_amd.ops.conv2d.forward")
    gen = torch.Generator(device).manual_seed(4)
    x, w = torch.randn(64, 256, 56, 56, generator=gen, device=device).bfloat16(), torch.randn(64, 256, 3, 3, generator=gen, device=device).bfloat16()
    args = (x, w, None, (1, 1), (1, 1), (1, 1))
    packed = [conv.conv2d_forward(*args) for _ in range(2)][-1]
    assert kernel._launch.conv(*args) is not None
    asked = []
    scratch = conv._scratch
    monkeypatch.setattr(conv, "_scratch", lambda nbytes, dev: asked.append(nbytes) or scratch(nbytes, dev))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(device).total_memory
    held = []
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (60 << 20)) / total)     # the result is 25 MB, the scratch 110
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                held.append(torch.empty(100 << 20, dtype=torch.uint8, device=device))                       # what the allocator keeps
        answered = kernel._launch.conv(*args) is not None
        bare = conv.conv2d_forward(*args)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert not answered
    assert asked and asked[0] > 100 << 20
    assert (bare.double() - packed.double()).norm() <= 2 ** -8 * packed.double().norm()
    assert torch.equal(conv.conv2d_forward(*args), packed) and len(asked) == 1                             # natively again
