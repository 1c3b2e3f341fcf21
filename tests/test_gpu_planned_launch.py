"""Repeated calls go through a kept launch (tritonix_amd/kernel.py: PlannedLaunch): it must see every change that the
long way sees -- other operands, an unaligned base, a replaced config, a hook -- and share nothing between threads."""
import threading

import pytest
import torch

import tritonix_amd.kernel as kernel
from tritonix_amd.ops import matmul as _  # noqa: F401
import importlib

mm = importlib.import_module("tritonix_amd.ops.matmul")
sg = importlib.import_module("tritonix_amd.ops.swiglu")

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def built_in_choice(monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    kernel._plans.clear()


def _ints(shape, dtype, seed):
    """Small integers: every product and sum is exact, whatever tile or split computes it."""
    g = torch.Generator("cpu").manual_seed(seed)
    return torch.randint(-4, 5, shape, generator=g).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.int8, torch.float32])
@pytest.mark.parametrize("m,n,k,layout", [(8, 520, 1024, "nn"), (65, 192, 100, "nn"), (128, 256, 64, "nt"), (72, 136, 128, "tn"),
                                          (1, 64, 320, "nn"), (16, 256, 4096, "nn")])
def test_repeated_calls_follow_their_operands(device, dtype, m, n, k, layout):
    for seed in range(3):                            # the first call binds, the next two take the kept launch
        a, b = _ints((m, k), dtype, 2 * seed), _ints((k, n), dtype, 2 * seed + 1)
        if dtype in (torch.float16, torch.bfloat16):
            b = b * (torch.arange(k).unsqueeze(1) % 4 == 0).to(dtype)
        ad = a.to(device) if layout != "tn" else a.t().contiguous().to(device).t()
        bd = b.to(device) if layout != "nt" else b.t().contiguous().to(device).t()
        want = a.double() @ b.double()
        for call in (mm.triton_matmul, mm.matmul_splitk):
            got = call(ad, bd)
            ref = want.to(got.dtype)
            assert got.shape == (m, n) and torch.equal(got.cpu(), ref), (call.__name__, seed)
    assert any(key[0] == "matmul" for key in kernel._plans)


def test_an_unaligned_operand_has_a_plan_of_its_own(device):
    store = torch.zeros(128 * 256 + 8, dtype=torch.float16, device=device)
    b = _ints((256, 128), torch.float16, 1).to(device)
    for off in (0, 1, 8, 3, 0):
        a = store[off:off + 128 * 256].view(128, 256)
        a.copy_(_ints((128, 256), torch.float16, off).to(device))
        assert torch.equal(mm.triton_matmul(a, b).cpu(), (a.cpu().double() @ b.cpu().double()).half())
    assert len([k for k in kernel._plans if k[0] == "matmul"]) == 2


def test_a_replaced_config_and_a_hook_are_seen(device):
    a, b = _ints((256, 128), torch.bfloat16, 0).to(device), _ints((128, 256), torch.bfloat16, 1).to(device)
    first = mm.triton_matmul(a, b)
    key = (256, 256, 128, torch.bfloat16, 1)
    mm._matmul_cfg[key] = dict(block_m=128, block_n=64, block_k=64, group_m=4, num_stages=3, num_warps=4)
    assert torch.equal(mm.triton_matmul(a, b), first)
    (plan, _), = [v for k, v in kernel._plans.items() if k[0] == "matmul"]
    assert (plan.template.block_m, plan.template.block_n) == (128, 64)
    seen = []
    mm.matmul_kernel.add_pre_run_hook(lambda *args, **kw: seen.append(kw["block_n"]))
    try:
        mm.triton_matmul(a, b)
    finally:
        mm.matmul_kernel.kernel.pre_run_hooks.clear()
    assert seen == [64]
    mm._matmul_cfg.pop(key)
    assert torch.equal(mm.triton_matmul(a, b), first) and key in mm._matmul_cfg


def test_activation_is_part_of_the_plan(device):
    x, w = torch.randn(32, 128, device=device).bfloat16(), torch.randn(128, 256, device=device).bfloat16() / 11
    out = {}
    for _ in range(2):
        for act in ("silu", "sigmoid", "none"):
            z = sg.glu(x, w, activation=act)
            assert torch.equal(out.setdefault(act, z), z)
    g, lin = (x.float() @ w.float())[:, 0::2], (x.float() @ w.float())[:, 1::2]
    for act, ref in (("silu", torch.nn.functional.silu(g) * lin), ("sigmoid", torch.sigmoid(g) * lin), ("none", g * lin)):
        # fp32 sums of 128 terms, one rounding to bf16
        assert (out[act].float() - ref).abs().max() <= 2 ** -8 * ref.abs().max() + 1e-3


def test_threads_with_streams_of_their_own_share_a_plan(device):
    a = [_ints((64, 2048), torch.float16, s).to(device) for s in range(4)]
    b = (_ints((2048, 256), torch.float16, 9) * (torch.arange(2048).unsqueeze(1) % 8 == 0).half()).to(device)
    want = [(x.cpu().double() @ b.cpu().double()).half() for x in a]
    mm.triton_matmul(a[0], b)
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                c = mm.triton_matmul(a[i], b)
                if not torch.equal(c.cpu(), want[i]):
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_a_size_met_once_costs_no_plan(device):
    """The first call of a size only notes it, the second keeps the launch, the third takes it."""
    a, b = _ints((24, 128), torch.float16, 0).to(device), _ints((128, 64), torch.float16, 1).to(device)
    first = mm.triton_matmul(a, b)
    assert list(kernel._plans.values()) == [None]
    second = mm.triton_matmul(a, b)
    (plan, _), = kernel._plans.values()
    assert isinstance(plan, kernel.PlannedLaunch)
    assert torch.equal(second, first) and torch.equal(mm.triton_matmul(a, b), first)
