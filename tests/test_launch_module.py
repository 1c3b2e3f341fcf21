"""tritonix_amd/_launch.so (csrc/launch.cpp): repeated calls without the interpreter.  It may answer only what the ordinary path
would do alike; everything else is None and goes the long way."""
import importlib
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch

import tritonix_amd.kernel as kernel

mm = importlib.import_module("tritonix_amd.ops.matmul")
sg = importlib.import_module("tritonix_amd.ops.swiglu")
conv = importlib.import_module("tritonix_amd.ops.conv2d.forward")


def test_it_is_built_and_answers_none_to_what_it_does_not_know():
    launch = kernel.launch_module()
    a, b = torch.zeros(4, 4), torch.zeros(4, 4)
    assert launch.product(0, a, b, {}, []) is None and launch.product(0, a, 3, {}, []) is None
    assert launch.conv(a, b, None, (1, 1), (0, 0), (1, 1)) is None
    with pytest.raises(ValueError):
        launch.keep(0, a, b, a, b"short", 0, 0, False, (), {})
    assert kernel.plan_tag("matmul") == 0 and kernel.plan_tag(("splitk", 4)) == kernel.plan_tag(("splitk", 4)) != 0


@pytest.fixture
def built_in(monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    kernel._plans.clear()


def _met(call, times=3):
    for _ in range(times):
        out = call()
    return out


@pytest.mark.gpu
def test_kept_calls_are_answered_natively_on_the_current_stream(built_in, device):
    a, b = torch.randn(40, 96, device=device).half(), torch.randn(96, 72, device=device).half()
    want = _met(lambda: mm.triton_matmul(a, b))
    hooks = mm.matmul_kernel.kernel.pre_run_hooks
    assert torch.equal(kernel._launch.product(0, a, b, mm._matmul_cfg, hooks), want)
    assert kernel._launch.product(0, a, b, mm._matmul_cfg, [print]) is None                     # a hook wants to see the call
    assert kernel._launch.product(0, a, b, {}, hooks) is None                                   # another config may be due
    assert kernel._launch.product(0, a, b.t().contiguous().t(), mm._matmul_cfg, hooks) is None  # other strides
    index = a.get_device()
    assert kernel._launch.stream_of(index) == kernel._stream_of(index)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert kernel._launch.stream_of(index) == kernel._stream_of(index) == side.cuda_stream
        got = mm.triton_matmul(a, b)
    side.synchronize()
    assert torch.equal(got, want)
    kernel._plans.clear()
    assert kernel._launch.product(0, a, b, mm._matmul_cfg, hooks) is None


@pytest.mark.gpu
def test_results_carry_no_gradient_and_wrapped_tensors_go_the_long_way(built_in, device):
    a = torch.nn.Parameter(torch.randn(24, 64, device=device).bfloat16())
    b = torch.randn(64, 40, device=device).bfloat16()
    out = _met(lambda: mm.triton_matmul(a, b))
    assert not out.requires_grad and torch.equal(out, mm.triton_matmul(a.detach(), b))
    hooks, seen = mm.matmul_kernel.kernel.pre_run_hooks, []

    def inner(x):
        seen.append(kernel._launch.product(0, x, b, mm._matmul_cfg, hooks))
        return x

    torch.vmap(inner)(torch.randn(3, 24, 64, device=device).bfloat16())
    assert seen == [None]


@pytest.mark.gpu
def test_split_gated_and_conv_calls(built_in, device):
    gen = torch.Generator(device).manual_seed(1)
    a, b = torch.randn(16, 4096, generator=gen, device=device).bfloat16(), torch.randn(4096, 256, generator=gen, device=device).bfloat16()
    first = mm.matmul_splitk(a, b)
    assert torch.equal(_met(lambda: mm.matmul_splitk(a, b), 4), first)
    assert torch.equal(_met(lambda: mm.matmul_splitk(a, b, split_k=8), 4), first)
    for act in ("silu", "sigmoid", "silu"):
        z = sg.glu(a, b, activation=act)
        assert torch.equal(_met(lambda: sg.glu(a, b, activation=act), 3), z)
    x = torch.randn(2, 24, 14, 14, generator=gen, device=device).half()
    w, bias = torch.randn(32, 24, 3, 3, generator=gen, device=device).half(), torch.randn(32, generator=gen, device=device).half()
    for args in ((x, w, bias), (x, w, None), (x, w, bias.float())):
        y = conv.conv2d_forward(*args, (1, 1), (1, 1), (1, 1))
        assert torch.equal(_met(lambda: conv.conv2d_forward(*args, (1, 1), (1, 1), (1, 1))), y)
        ref = torch.nn.functional.conv2d(x.double(), w.double(), None if args[2] is None else args[2].double(), padding=1)
        assert (y.double() - ref).norm() <= 2 ** -10 * ref.norm()
    with pytest.raises(AssertionError):
        conv.conv2d_forward(x.transpose(2, 3), w, bias, (1, 1), (1, 1), (1, 1))


@pytest.mark.gpu
def test_threads_repeat_kept_calls_on_streams_of_their_own(built_in, device):
    """The interpreter lock is given back around the launch, so calls of several threads interleave there: same bits, plans kept
    and dropped meanwhile."""
    gen = torch.Generator(device).manual_seed(2)
    a, b = torch.randn(16, 4096, generator=gen, device=device).bfloat16(), torch.randn(4096, 256, generator=gen, device=device).bfloat16()
    f, g = torch.randn(300, 640, generator=gen, device=device), torch.randn(640, 320, generator=gen, device=device)
    x, w = torch.randn(2, 24, 14, 14, generator=gen, device=device).half(), torch.randn(32, 24, 3, 3, generator=gen, device=device).half()
    calls = [lambda: mm.matmul_splitk(a, b), lambda: mm.triton_matmul(f, g), lambda: conv.conv2d_forward(x, w, None, (1, 1), (1, 1), (1, 1))]
    want = [_met(c) for c in calls]
    torch.cuda.synchronize()

    def work(turn):
        stream, wrong = torch.cuda.Stream(device), 0
        with torch.cuda.stream(stream):
            for i in range(60):
                got = calls[(turn + i) % 3]()
                stream.synchronize()
                wrong += not torch.equal(got, want[(turn + i) % 3])
                if turn == 0 and i % 20 == 10:
                    kernel._plans.clear()
        return wrong

    with ThreadPoolExecutor(4) as pool:
        assert list(pool.map(work, range(4))) == [0] * 4
