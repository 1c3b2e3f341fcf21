"""Launch objects that keep the reference's Triton calling convention over the HIP engine.

A reference kernel is launched as ``kernel[grid](a, b, c, m, n, k, stride_am,
stride_ak, stride_bk, stride_bn, stride_cm, stride_cn, block_m=..., block_n=...,
block_k=..., group_m=..., [split_k=...,] num_stages=..., num_warps=...)``
(tritonix/ops/matmul.py:222-236, :249-263; the GLU kernel adds ``use_tf32``
and ``activation``, tritonix/ops/swiglu.py:24-43).  ``HipKernel`` accepts the
same call, turns it into one ``tnx_gemm`` through the C ABI and launches on
torch's current stream.  ``grid`` is accepted for compatibility; the engine
derives its own 1-D grid from the shape and the tile.
"""
from __future__ import annotations

import ctypes
import itertools
import threading
import warnings
from collections import OrderedDict
from typing import Callable, List, Optional, Tuple

from tritonix_amd import _C

__all__ = ["HipKernel", "cdiv"]


def cdiv(a: int, b: int) -> int:
    return -(-a // b)


_POSITIONAL = ("a", "b", "c", "m", "n", "k", "stride_am", "stride_ak", "stride_bk", "stride_bn", "stride_cm",
               "stride_cn")
_ACTIVATIONS = {"silu": _C.EPI_GLU_SILU, "sigmoid": _C.EPI_GLU_SIGMOID}

# split-K scratch buffers, most recently used last; at most _MAX_WORKSPACES are kept alive
_workspaces: "OrderedDict[Tuple[int, int], object]" = OrderedDict()
_workspaces_lock = threading.RLock()           # (an allocation may run other Python code of its thread)
_MAX_WORKSPACES = 8


def _torch_dtype_code(dtype) -> int:
    import torch

    table = {torch.float16: _C.F16, torch.bfloat16: _C.BF16, torch.int8: _C.I8, torch.int32: _C.I32,
             torch.float32: _C.F32}
    if dtype not in table:
        raise ValueError(f"dtype {dtype} has no HIP kernel (float16, bfloat16, int8 and -- as a bf16 split -- float32 inputs are built)")
    return table[dtype]


def out_dtype_for(dtype):
    """Output dtype of the engine for an input dtype: floats keep theirs, int8 accumulates to int32."""
    import torch

    return torch.int32 if dtype == torch.int8 else dtype


def _workspace_key(device, stream_ptr: int, atomic: bool = False) -> Tuple[int, int, bool]:
    import torch

    return (device.index if device.index is not None else torch.cuda.current_device(), stream_ptr, bool(atomic))


def _workspace(device, stream_ptr: int, nbytes: int, atomic: bool = False):
    """Split-K scratch, one growing buffer per (device, stream), the least recently used ones released.

    Allocated zero-filled: the leading counter region must start at zero and every launch leaves it zero.  A
    launch that fails part-way may leave counters set, so ``drop_workspace`` forgets the buffer after any error
    and the next launch starts from a freshly zeroed one.
    """
    import torch

    # launches that reduce with atomics need their sum region zero and leave it zero; ordered launches leave
    # slices behind: the two modes never share a buffer
    key = _workspace_key(device, stream_ptr, atomic)
    with _workspaces_lock:              # a thread that evicts between another one's lookup and its move to the end
        buf = _workspaces.get(key)
        if buf is None or buf.numel() < nbytes:
            buf = torch.zeros(max(nbytes, 1 << 20), dtype=torch.uint8, device=device)
            _workspaces[key] = buf
        _workspaces.move_to_end(key)
        if _capturing():
            # A launch recorded into a HIP graph bakes this pointer into the graph: the buffer must outlive every
            # replay, so it is never released (not by the eviction below, not when a later call needs a larger one).
            if not any(kept is buf for kept in _captured_workspaces):
                _captured_workspaces.append(buf)
            return buf
        while len(_workspaces) > _MAX_WORKSPACES:
            _workspaces.popitem(last=False)       # launches already enqueued keep their buffer alive through the allocator's stream ordering
        return buf


# scratch buffers handed to launches that were recorded into a HIP graph: alive until the process ends
_captured_workspaces: list = []


def _capturing() -> bool:
    import torch

    try:
        return bool(torch.cuda.is_current_stream_capturing())
    except (RuntimeError, AssertionError):
        return False


def drop_workspace(device, stream_ptr: int) -> None:
    """Forget the scratch of (device, stream): called when a launch on it reported an error."""
    with _workspaces_lock:
        for atomic in (False, True):
            _workspaces.pop(_workspace_key(device, stream_ptr, atomic), None)


def _stream_of(index: int) -> int:
    """Handle of torch's current stream on a device, without the stream object (0.2 us instead of 1.2)."""
    import torch

    try:
        return torch._C._cuda_getCurrentRawStream(index)
    except AttributeError:
        return torch.cuda.current_stream(index).cuda_stream


class PlannedLaunch:
    """A launch that went through ``HipKernel.run`` once, kept by what it depends on -- sizes, strides, types, device,
    tile -- and none of its pointers: repeating it fills those in.

    Binding every argument by name, checking it, and asking the library for scratch sizes anew took 21 us of host time
    per product, four times what a small one (1024 x 768 x 512, 5 us) takes on the GPU."""

    __slots__ = ("kernel", "template", "shape", "dtype", "index", "scratch", "slices", "atomic", "lib", "cfg")

    def __init__(self, kernel: "HipKernel", a, b, c, cfg: dict, extra: dict):
        self.kernel, self.cfg = kernel, dict(cfg)
        bound = dict(zip(_POSITIONAL, (a, b, c, a.shape[0], b.shape[1], a.shape[1], *a.stride(), *b.stride(), *c.stride())))
        g = kernel.make_args({**bound, **cfg, **extra})
        g.a = g.b = g.c = None
        self.template, self.shape, self.dtype, self.index = g, tuple(c.shape), c.dtype, a.get_device()
        self.lib = lib = _C.load()
        self.scratch = int(lib.tnx_gemm_f32_scratch_bytes(ctypes.byref(g))) if g.in_dtype == _C.F32 else 0
        self.slices = int(lib.tnx_gemm_workspace_bytes(ctypes.byref(g))) if g.split_k > 1 else 0
        self.atomic = bool(g.schedule & _C.SCHED_ATOMIC_REDUCE)

    def __call__(self, a, b):
        import torch

        device = a.device
        c = torch.empty(self.shape, device=device, dtype=self.dtype)
        g = _C.GemmArgs.from_buffer_copy(self.template)       # its own copy: threads share the template
        g.a, g.b, g.c = a.data_ptr(), b.data_ptr(), c.data_ptr()
        if self.index != torch.cuda.current_device():
            with torch.cuda.device(device):
                status = self._go(g, device)
        else:
            status = self._go(g, device)
        if status:
            _C.raise_for_status(status, g)
        return c

    def _go(self, g, device) -> int:
        stream = g.stream = _stream_of(self.index)
        if self.slices:
            ws = _workspace(device, stream, self.slices, self.atomic)
            g.workspace, g.workspace_bytes = ws.data_ptr(), ws.numel()
        if g.in_dtype == _C.F32:
            import torch

            scratch = torch.empty(self.scratch, dtype=torch.uint8, device=device) if self.scratch else None
            status = self.lib.tnx_gemm_f32(ctypes.byref(g), scratch.data_ptr() if self.scratch else None, self.scratch)
            g.in_dtype = _C.BF16 if status else g.in_dtype          # what an error message has to describe
        else:
            status = self.lib.tnx_gemm(ctypes.byref(g))
        if status == _C.E_HIP and g.split_k > 1:
            drop_workspace(device, stream)
        return status


class _Plans(dict):
    """The kept launches; what the native side holds of them goes with them."""

    def clear(self) -> None:
        super().clear()
        if _launch is not None:
            _launch.forget()


# by everything a launch depends on but its pointers (None: met once so far); bounded, dropped whole when full
_plans: dict = _Plans()
_MAX_PLANS = 1024

# tritonix_amd/_launch.so (csrc/launch.cpp), which repeats a kept launch without the interpreter; loaded with the first of them
_launch = None
_launch_missing = False
_tags: dict = {"matmul": 0}
_tag_numbers = itertools.count(1)
_tags_lock = threading.Lock()


def product(tag: int, a, b, memo: dict, hooks: list):
    """The product of ``a`` and ``b`` by a kept launch of the native side, or None.  (Replaced by ``_launch.product`` once there
    is such a launch.)"""
    return None


def plan_tag(tag) -> int:
    """A number for the operation of a plan key, never another one's: not where threads ask at once, and not after the tags have
    been dropped, when a thread may still hold an old number."""
    n = _tags.get(tag)
    if n is None:
        with _tags_lock:
            n = _tags.get(tag)
            if n is None:
                if len(_tags) >= _MAX_PLANS:
                    _plans.clear()
                    _tags.clear()
                    _tags["matmul"] = 0
                n = _tags[tag] = next(_tag_numbers)
    return n


def _workspace_of(index: int, stream: int, nbytes: int, atomic: int):
    """The buffer itself, for the caller to hold until its launch is queued."""
    import torch

    return _workspace(torch.device("cuda", index), stream, nbytes, bool(atomic))


def _launch_failed(index: int, stream: int, status: int, args: bytes) -> None:
    """What ``PlannedLaunch`` does about a launch that reported an error."""
    import torch

    g = _C.GemmArgs.from_buffer_copy(args)
    if status == _C.E_HIP and g.split_k > 1:
        drop_workspace(torch.device("cuda", index), stream)
    g.in_dtype = _C.BF16 if g.in_dtype == _C.F32 else g.in_dtype
    _C.raise_for_status(status, g)


def launch_module():
    """``_launch``, bound to the loaded library, or None where it was not built or was built against another torch: it only
    repeats what the ordinary path does, which then takes every call."""
    global _launch, product, _launch_missing
    if _launch is None and not _launch_missing:
        try:
            import torch
            from tritonix_amd import _launch as module

            if module.torch_version != torch.__version__.split("+")[0]:
                raise ImportError(f"built against torch {module.torch_version}, this is {torch.__version__}")
        except (ImportError, AttributeError) as err:
            _launch_missing = True
            warnings.warn(f"tritonix_amd/_launch.so cannot be used ({err}): repeated calls take the interpreter's path, a few "
                          "microseconds longer; `python -m tritonix_amd.build` builds it", RuntimeWarning, stacklevel=2)
            return None
        _bind(module, _C.load().tnx_gemm)
        _launch, product = module, module.product
    return _launch


def _bind(module, gemm, workspace=_workspace_of) -> None:
    """Hand the native side its entry points: the library's, with ``gemm`` for 16-bit and int8 products."""
    lib = _C.load()
    module.bind(*(ctypes.cast(fn, ctypes.c_void_p).value for fn in (gemm, lib.tnx_gemm_f32, lib.tnx_conv2d_forward)), workspace, _launch_failed)


def plan_key(tag, a, b) -> tuple:
    """What a product of ``a`` and ``b`` depends on: sizes, strides, types, devices, and whether the base pointers are
    16-byte aligned (which decides between the loaders)."""
    return (tag, a.shape, b.shape, a.stride(), b.stride(), a.dtype, b.dtype, a.get_device(), b.get_device(),
            (a.data_ptr() | b.data_ptr()) & 15 == 0)


def planned(key: tuple, memo: dict) -> Optional[PlannedLaunch]:
    """The launch kept for ``key`` -- unless the config memo now holds another tile for it, or a hook wants to see the call."""
    hit = _plans.get(key)
    if hit is None or hit[0].kernel.pre_run_hooks or memo.get(hit[1]) != hit[0].cfg:
        return None
    return hit[0]


def keep_plan(key: tuple, memo_key: tuple, memo: dict, kernel, a, b, c, given, **extra) -> None:
    """Operands that had to be copied first keep the long way; views of the ``given`` ones (a row with another pitch) do not.
    Remember the launch that just gave ``c``, the second time it is met: making it ready takes 9 us, which a program that
    never meets a size twice would pay for nothing (first call of a 16-bit product 34 us with it, 26 without)."""
    if a.data_ptr() != given[0].data_ptr() or b.data_ptr() != given[1].data_ptr():
        return
    if key not in _plans:
        if len(_plans) >= _MAX_PLANS:
            _plans.clear()
        _plans[key] = None
        return
    kernel = getattr(kernel, "kernel", kernel)                # the launch object behind its tunable wrapper
    if a.get_device() < 0 or memo_key not in memo or not isinstance(kernel, HipKernel):
        return
    plan = PlannedLaunch(kernel, a, b, c, memo[memo_key], extra)
    _plans[key] = (plan, memo_key)
    native = launch_module()
    if native is not None:
        native.keep(plan_tag(key[0]), *given, c, bytes(plan.template), plan.scratch, plan.slices, plan.atomic, memo_key, plan.cfg)


class _BoundLaunch:
    def __init__(self, kernel: "HipKernel", grid):
        self.kernel, self.grid = kernel, grid

    def __call__(self, *args, **kwargs):
        return self.kernel.run(*args, grid=self.grid, **kwargs)


class HipKernel:
    """One entry of the HIP engine behind the Triton launch protocol."""

    def __init__(self, name: str, tile_params: List[str], glu: bool = False, doc: Optional[str] = None):
        self.__name__ = name
        self.__doc__ = doc
        self.tile_params = list(tile_params)
        self.glu = glu
        # optional keywords after the reference's own: a K split for kernels whose signature has none, the
        # number of trailing tiles the split applies to (0 = all), and the two scheduling switches of the engine
        # (persistent: one workgroup per CU walks its tiles; superblock: 16x16 super-block launch order)
        # atomic_reduce: split-K slices are added into one fp32 copy with atomics instead of being summed in order
        self.optional = [n for n in ("split_k", "tail_tiles", "persistent", "superblock", "atomic_reduce")
                         if n not in self.tile_params]
        self.arg_names = (list(_POSITIONAL) + self.tile_params + (["use_tf32", "activation"] if glu else [])
                          + self.optional)
        self.pre_run_hooks: List[Callable] = []
        self.specialize_keys: List[str] = []

    def __getitem__(self, grid) -> _BoundLaunch:
        return _BoundLaunch(self, grid)

    def add_pre_run_hook(self, hook: Callable) -> None:
        """``hook(*args, **kwargs)`` runs before every launch, as with a Triton ``JITFunction``."""
        self.pre_run_hooks.append(hook)

    # ------------------------------------------------------------------
    def _bind(self, args, kwargs) -> dict:
        if len(args) > len(self.arg_names):
            raise TypeError(f"{self.__name__} takes at most {len(self.arg_names)} arguments, got {len(args)}")
        bound = dict(zip(self.arg_names, args))
        for k, v in kwargs.items():
            if k not in self.arg_names:
                raise TypeError(f"{self.__name__} got an unexpected keyword argument '{k}'")
            if k in bound:
                raise TypeError(f"{self.__name__} got multiple values for argument '{k}'")
            bound[k] = v
        missing = [n for n in list(_POSITIONAL) + self.tile_params if n not in bound]
        if missing:
            raise TypeError(f"{self.__name__} missing arguments: {', '.join(missing)}")
        return bound

    def make_args(self, bound: dict) -> _C.GemmArgs:
        """Fill a ``tnx_gemm_args`` from a bound call (pointers from the tensors' ``data_ptr``)."""
        a, b, c = bound["a"], bound["b"], bound["c"]
        g = _C.GemmArgs()
        g.a, g.b, g.c = a.data_ptr(), b.data_ptr(), c.data_ptr()
        g.m, g.n, g.k = int(bound["m"]), int(bound["n"]), int(bound["k"])
        g.stride_am, g.stride_ak = int(bound["stride_am"]), int(bound["stride_ak"])
        g.stride_bk, g.stride_bn = int(bound["stride_bk"]), int(bound["stride_bn"])
        g.stride_cm, g.stride_cn = int(bound["stride_cm"]), int(bound["stride_cn"])
        g.in_dtype = _torch_dtype_code(a.dtype)
        if b.dtype != a.dtype:
            raise ValueError(f"a and b must share a dtype, got {a.dtype} and {b.dtype}")
        g.out_dtype = _torch_dtype_code(c.dtype)
        g.block_m, g.block_n, g.block_k = int(bound["block_m"]), int(bound["block_n"]), int(bound["block_k"])
        g.group_m = int(bound["group_m"])
        g.split_k = int(bound.get("split_k", 1))
        g.tail_tiles = int(bound.get("tail_tiles", 0))
        g.schedule = ((_C.SCHED_PERSISTENT if int(bound.get("persistent", 0)) else 0)
                      | (_C.SCHED_SUPERBLOCK if int(bound.get("superblock", 0)) else 0)
                      | (_C.SCHED_ATOMIC_REDUCE if int(bound.get("atomic_reduce", 0)) else 0))
        g.num_stages, g.num_warps = int(bound["num_stages"]), int(bound["num_warps"])
        if self.glu:
            # "silu" and "sigmoid" gate explicitly; like the reference kernel, any other
            # value leaves the gate un-activated (tritonix/ops/swiglu.py:100-102)
            g.epilogue = _ACTIVATIONS.get(bound.get("activation", "silu"), _C.EPI_GLU_IDENTITY)
        else:
            g.epilogue = _C.EPI_NONE
        return g

    def run(self, *args, grid=None, **kwargs):
        import torch

        bound = self._bind(args, kwargs)
        a, b, c = bound["a"], bound["b"], bound["c"]
        for name, t in (("a", a), ("b", b), ("c", c)):
            if not isinstance(t, torch.Tensor) or not t.is_cuda:
                raise ValueError(f"{self.__name__}: '{name}' must be a tensor on a HIP device")
        if not (a.device == b.device == c.device):
            raise ValueError(f"{self.__name__}: a, b and c must live on one device")
        if grid is not None and not callable(grid):
            if not all(isinstance(g, int) and g >= 0 for g in tuple(grid)):
                raise ValueError(f"{self.__name__}: grid must be a tuple of non-negative ints, got {grid!r}")
        for hook in self.pre_run_hooks:
            hook(*args, **kwargs)

        lib = _C.load()
        if a.dtype == torch.float32 and b.dtype == torch.float32:
            if c.dtype != torch.float32:
                raise ValueError(f"{self.__name__}: float32 operands give a float32 result, got c of {c.dtype}")
        g = self.make_args(bound)
        if a.device.index != torch.cuda.current_device():
            with torch.cuda.device(a.device):
                status = self._launch(lib, g, a.device)
        else:
            status = self._launch(lib, g, a.device)
        _C.raise_for_status(status, g)
        return None

    @staticmethod
    def _launch(lib, g, device) -> int:
        import torch

        stream = torch.cuda.current_stream(device).cuda_stream
        g.stream = stream
        scratch = None
        if g.in_dtype == _C.F32:
            # the reference's kernels take float32 operands and multiply them in TF32 (tritonix/ops/matmul.py:98,
            # tritonix/ops/swiglu.py:89-93), for which gfx950 has no matrix instruction: the library cuts them into bf16
            # heads and tails and multiplies those, with a float32 result
            # -- or, for small products and few rows, multiplies them as they are, without scratch
            need = int(lib.tnx_gemm_f32_scratch_bytes(ctypes.byref(g)))
            scratch = torch.empty(need, dtype=torch.uint8, device=device)
        if g.split_k > 1:
            need = int(lib.tnx_gemm_workspace_bytes(ctypes.byref(g)))
            if need:
                ws = _workspace(device, stream, need, bool(g.schedule & _C.SCHED_ATOMIC_REDUCE))
                g.workspace, g.workspace_bytes = ws.data_ptr(), ws.numel()
        if scratch is None:
            status = lib.tnx_gemm(ctypes.byref(g))
        else:
            status = lib.tnx_gemm_f32(ctypes.byref(g), scratch.data_ptr(), scratch.numel())
            g.in_dtype = _C.BF16 if status else g.in_dtype          # what an error message has to describe
        if status == _C.E_HIP and g.split_k > 1:
            drop_workspace(device, stream)
        return status

    def prepare(self, *args, **kwargs) -> Callable[[], None]:
        """Bind a launch once and return a zero-argument callable that repeats it.

        The tensors, tile config, stream and split-K workspace are captured at bind time; the returned
        callable only performs the C-ABI call (for launch-bound shapes and for benchmarks).
        """
        import torch

        bound = self._bind(args, kwargs)
        lib = _C.load()
        if bound["a"].dtype == torch.float32:
            raise ValueError(f"{self.__name__}.prepare binds 16-bit and int8 launches; a float32 call splits its operands "
                             "on every launch")
        g = self.make_args(bound)
        device = bound["a"].device
        stream = torch.cuda.current_stream(device).cuda_stream
        g.stream = stream
        keep = [bound["a"], bound["b"], bound["c"]]
        if g.split_k > 1:
            need = int(lib.tnx_gemm_workspace_bytes(ctypes.byref(g)))
            ws = _workspace(device, stream, need, bool(g.schedule & _C.SCHED_ATOMIC_REDUCE))
            g.workspace, g.workspace_bytes = ws.data_ptr(), ws.numel()
            keep.append(ws)
        status = lib.tnx_gemm_supported(ctypes.byref(g))
        _C.raise_for_status(status, g)
        ref, fn = ctypes.byref(g), lib.tnx_gemm

        def launch(_keep=keep, _g=g):
            st = fn(ref)
            if st:
                if _g.split_k > 1:
                    drop_workspace(device, stream)
                _C.raise_for_status(st, _g)

        return launch

    # host-only helpers -------------------------------------------------
    def lds_bytes(self, in_dtype_code: int, block_m: int, block_n: int, block_k: int, num_stages: int,
                  num_warps: int = 4, persistent: int = 0) -> int:
        """LDS bytes per workgroup of a tile config (no GPU needed)."""
        g = _C.GemmArgs()
        g.in_dtype = in_dtype_code
        g.block_m, g.block_n, g.block_k, g.num_stages, g.num_warps = block_m, block_n, block_k, num_stages, num_warps
        g.schedule = _C.SCHED_PERSISTENT if persistent else 0
        return int(_C.load().tnx_gemm_lds_bytes(ctypes.byref(g)))

    def __repr__(self):
        return f"<HipKernel {self.__name__}>"
