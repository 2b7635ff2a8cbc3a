"""Launchers: the same four names and argument meaning as the forward launchers
of the reference (``grouped_mm_bf16/kernels.py:524-717``) -- each writes into a
caller-allocated ``out`` and returns None -- but they hand raw pointers, sizes
and strides to the gfx950 kernels behind the C ABI instead of JIT-compiling
Triton.  ``out.dtype`` selects the epilogue (input dtype or float32), as the
reference's ``OUT_DTYPE=_as_tl_dtype(out.dtype)`` does.

The launch itself is registered as the torch custom op
``grouped_mm_bf16_amd::launch`` (mutating ``out``) so that it is visible to
torch's dispatcher and tracing; it runs on the current stream of the operands'
device and never synchronises.
"""
from __future__ import annotations

import contextlib
from typing import Optional

import torch

from . import _lib

_DTYPE_CODE = {torch.bfloat16: _lib.DT_BF16, torch.float16: _lib.DT_F16, torch.float32: _lib.DT_F32}

V_2D3D, V_3D3D, V_2D2D, V_3D2D = 0, 1, 2, 3


def _dtype_code(dtype: torch.dtype) -> int:
    try:
        return _DTYPE_CODE[dtype]
    except KeyError:
        raise RuntimeError(f"Unsupported dtype: {dtype}") from None


def _require_gpu(*tensors) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("grouped_mm_bf16 is GPU-only (CUDA/HIP); CPU tensors are not supported")


def current_stream(device: torch.device) -> int:
    """Handle of torch's current stream of `device`.  ``torch.cuda.current_stream().cuda_stream`` builds a Stream object
    for it: 2.6 us of a 17 us call, this 0.1 us."""
    return torch._C._cuda_getCurrentRawStream(device.index)


# The same for torch.cuda.current_device(), which first makes sure that there is a device: here a tensor lies on it.
current_device = getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device)


# One workspace per (device, stream): launches on one stream run one after the other, so they can share it;
# launches on different streams may overlap and must not.  Allocated on first use and kept (the library leaves
# the arrival counters at its head zero after every launch).  For eager launches only: a captured launch runs on
# whatever stream its graph is replayed on, beside anything else.
_workspaces: dict = {}

_EAGER_ONLY = _lib.WORKSPACE_EAGER_ONLY

# Last capture seen: its id, and whether torch gives allocations made inside it to the graph.
_capture = (0, False)


def workspace(device: torch.device, stream: int):
    """(pointer, bytes) of the workspace for eager launches on `stream` of `device`, or (None, 0) when none can be
    had."""
    key = (device.index, stream)
    ws = _workspaces.get(key)
    if ws is None:
        nbytes = _lib.load().gmm_workspace_bytes()
        if nbytes <= 0 or torch.cuda.is_current_stream_capturing():
            return None, 0
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=device)
        _workspaces[key] = ws
    return ws.data_ptr(), ws.numel()


def _captured_workspace(device: torch.device, stream: int) -> Optional[torch.Tensor]:
    """A workspace for one launch inside a capture: allocated and cleared there, so that it belongs to the graph's memory
    pool, which nothing but the graph uses (later allocations of the capture may share the memory: they follow on the
    same stream).  None in a capture that torch does not know of: memory allocated there would go back to the common
    pool."""
    global _capture
    lib = _lib.load()
    capture = lib.gmm_stream_capture(stream)
    known, owned = _capture
    if capture != known:
        # torch's ordinary allocations lie in pool (0, 0)
        probe = torch.empty(1, device=device).data_ptr()
        owned = any(s["address"] <= probe < s["address"] + s["total_size"] and tuple(s["segment_pool_id"]) != (0, 0)
                    for s in torch.cuda.memory_snapshot() if s["device"] == device.index)
        _capture = capture, owned
    if not owned:
        return None
    ws = torch.empty(lib.gmm_workspace_bytes(), dtype=torch.uint8, device=device)
    ws[:4096].zero_()
    return ws


def call_with_workspace(launcher, args: tuple, device: torch.device, stream: int) -> int:
    """``launcher(*args, workspace, workspace_bytes, stream)`` with the stream's workspace, or with one of its own inside a
    capture if the launch has a use for it; returns the status."""
    ws = _workspaces.get((device.index, stream))     # as workspace() has it, without the call
    if ws is not None:
        rc = launcher(*args, ws.data_ptr(), ws.numel() | _EAGER_ONLY, stream)
    else:
        ws, nbytes = workspace(device, stream)
        rc = launcher(*args, ws, nbytes | _EAGER_ONLY, stream)
    if rc != _lib.ERR_WORKSPACE:
        return rc
    own = _captured_workspace(device, stream)
    if own is None:
        return launcher(*args, None, 0, stream)
    return launcher(*args, own.data_ptr(), own.numel(), stream)


def _launch_now(variant: int, a: torch.Tensor, b: torch.Tensor, offs: Optional[torch.Tensor],
                out: torch.Tensor) -> None:
    lib = _lib.load()
    _require_gpu(a, b, offs, out)
    device = a.device
    # the device guard costs microseconds; only switch when the tensors live on another device
    if device.index != current_device():
        with torch.cuda.device(device):
            _launch_here(lib, device, variant, a, b, offs, out)
    else:
        _launch_here(lib, device, variant, a, b, offs, out)


def _launch_here(lib, device: torch.device, variant: int, a: torch.Tensor, b: torch.Tensor, offs: Optional[torch.Tensor],
                 out: torch.Tensor) -> None:
    in_dt, out_dt = _dtype_code(a.dtype), _dtype_code(out.dtype)
    stream = current_stream(device)
    pa, pb, po = a.data_ptr(), b.data_ptr(), out.data_ptr()
    poffs = offs.data_ptr() if offs is not None else None
    if variant == V_2D3D:
        launcher = lib.gmm_2d3d
        args = (pa, pb, po, poffs, offs.numel(), a.size(0), b.size(2), a.size(1),
                a.stride(0), a.stride(1), b.stride(0), b.stride(1), b.stride(2),
                out.stride(0), out.stride(1), in_dt, out_dt)
    elif variant == V_3D3D:
        launcher = lib.gmm_3d3d
        args = (pa, pb, po, a.size(0), a.size(1), b.size(2), a.size(2),
                a.stride(0), a.stride(1), a.stride(2), b.stride(0), b.stride(1), b.stride(2),
                out.stride(0), out.stride(1), out.stride(2), in_dt, out_dt)
    elif variant == V_2D2D:
        launcher = lib.gmm_2d2d
        args = (pa, pb, po, poffs, offs.numel(), a.size(0), b.size(1), a.size(1),
                a.stride(0), a.stride(1), b.stride(0), b.stride(1),
                out.stride(0), out.stride(1), out.stride(2), in_dt, out_dt)
    elif variant == V_3D2D:
        launcher = lib.gmm_3d2d
        args = (pa, pb, po, poffs, offs.numel(), a.size(1), b.size(1), a.size(2),
                a.stride(0), a.stride(1), a.stride(2), b.stride(0), b.stride(1),
                out.stride(0), out.stride(1), in_dt, out_dt)
    else:
        raise RuntimeError(f"unknown variant {variant}")
    rc = call_with_workspace(launcher, args, device, stream)
    _lib.check(rc, "grouped_mm launch")


# The launch as a torch custom op (mutates `out`), for callers that trace or compile.  Eager calls skip
# the dispatcher, which costs more than the kernel for small products.
_launch_op = torch.library.custom_op("grouped_mm_bf16_amd::launch", mutates_args=("out",))(_launch_now)


@_launch_op.register_fake
def _launch_fake(variant, a, b, offs, out) -> None:
    """Shape propagation under FakeTensor: the op returns nothing and only fills `out`."""
    return None


def _launch(variant: int, a: torch.Tensor, b: torch.Tensor, offs: Optional[torch.Tensor], out: torch.Tensor) -> None:
    if torch.compiler.is_compiling():
        _launch_op(variant, a, b, offs, out)
    else:
        _launch_now(variant, a, b, offs, out)


# Bytes from which a gradient is not cleared first: torch's fill of 32 MiB takes as long as the kernel that looks at the offsets
# (5 us; 134 MB 18.5), and a smaller one costs less host time than that launch.
_CLEAR_FIRST_BELOW = 32 << 20


def launch_zeroed(variant: int, a: torch.Tensor, b: torch.Tensor, offs: torch.Tensor, shape) -> torch.Tensor:
    """A new tensor with the product of a variant with jagged rows or columns in it, zeros where no group owns anything: what a
    gradient has to be.  A large one is not cleared as a whole, which wrote it twice."""
    if torch.compiler.is_compiling() or shape[0] * shape[1] * a.element_size() < _CLEAR_FIRST_BELOW:
        out = torch.zeros(shape, device=a.device, dtype=a.dtype)
        if out.numel():
            _launch(variant, a, b, offs, out)
        return out
    out = torch.empty(shape, device=a.device, dtype=a.dtype)
    _launch_now(variant, a, b, offs, out)
    _zero_unowned(out, offs, variant == V_3D2D)
    return out


def _zero_unowned(out: torch.Tensor, offs: torch.Tensor, by_columns: bool) -> None:
    with torch.cuda.device(out.device) if out.device.index != current_device() else contextlib.nullcontext():
        rc = _lib.load().gmm_zero_unowned(out.data_ptr(), offs.data_ptr(), offs.numel(), int(by_columns), out.size(0), out.size(1),
                                          out.stride(0), out.stride(1), _dtype_code(out.dtype), current_stream(out.device))
    _lib.check(rc, "zeros past the last offset")


def grouped_mm_3d3d(mat_a: torch.Tensor, mat_b: torch.Tensor, out: torch.Tensor) -> None:
    """out[g] = mat_a[g] @ mat_b[g]  (reference ``kernels.py:524-550``)."""
    if mat_a.size(0) != mat_b.size(0):
        raise RuntimeError("batched dimension has to match")
    _launch(V_3D3D, mat_a, mat_b, None, out)


def grouped_mm_2d2d(mat_a: torch.Tensor, mat_b: torch.Tensor, offs: torch.Tensor, out: torch.Tensor) -> None:
    """out[g] = mat_a[:, s_g:e_g] @ mat_b[s_g:e_g, :], zeros for an empty group
    (reference ``kernels.py:553-580``)."""
    _launch(V_2D2D, mat_a, mat_b, offs, out)


def grouped_mm_2d3d(mat_a: torch.Tensor, mat_b: torch.Tensor, offs: torch.Tensor, out: torch.Tensor) -> None:
    """out[s_g:e_g] = mat_a[s_g:e_g] @ mat_b[g]  (reference ``kernels.py:583-686``)."""
    if offs.numel() != mat_b.size(0):
        raise RuntimeError("matrix batch sizes have to match")
    if mat_a.size(0) == 0 or mat_b.size(2) == 0:
        return
    _launch(V_2D3D, mat_a, mat_b, offs, out)


def grouped_mm_3d2d(mat_a: torch.Tensor, mat_b: torch.Tensor, offs: torch.Tensor, out: torch.Tensor) -> None:
    """out[:, s_g:e_g] = mat_a[g] @ mat_b[:, s_g:e_g]  (reference ``kernels.py:689-717``)."""
    if offs.numel() != mat_a.size(0):
        raise RuntimeError("matrix batch sizes have to match")
    _launch(V_3D2D, mat_a, mat_b, offs, out)


# ---- test / tuning hooks ---------------------------------------------------- #
@contextlib.contextmanager
def forced_path(path: str):
    """Force a kernel family ("auto", "generic" or "mfma") inside the block.

    The reference's tests force tile sizes through environment variables
    (``tests/test_grouped_mm.py:388-394``); this is the equivalent hook here.
    """
    code = {"auto": _lib.PATH_AUTO, "generic": _lib.PATH_GENERIC, "mfma": _lib.PATH_MFMA}[path]
    lib = _lib.load()
    prev = lib.gmm_set_path(code)
    try:
        yield
    finally:
        lib.gmm_set_path(prev)


@contextlib.contextmanager
def forced_mfma_config(config: int):
    lib = _lib.load()
    prev = lib.gmm_set_mfma_config(config)
    try:
        yield
    finally:
        lib.gmm_set_mfma_config(prev)


@contextlib.contextmanager
def forced_tile_heights(tall: int, shrt: int):
    """Force the tile heights of the assembly tile (tall 256 / 128, short 64 / 0; -1 = automatic)."""
    lib = _lib.load()
    prev = lib.gmm_set_tile_heights(tall, shrt)   # ((tall + 1) << 16) | (short + 1) of the previous setting
    try:
        yield
    finally:
        lib.gmm_set_tile_heights((prev >> 16) - 1, (prev & 0xffff) - 1)


@contextlib.contextmanager
def tail_split(on: bool):
    """Inside the block launches do (True) or do not (False) use their workspace: cut the tiles of a sparse last round or the
    groups of a jagged contraction along the contraction, draw tiles from its counters.  A cut tile adds its fp32 partial sums in a fixed order, so results are reproducible either
    way, but they differ in the last bit from the uncut tile's: tests that compare two launches bit for bit
    across different tile lists switch the split off."""
    lib = _lib.load()
    prev = lib.gmm_set_tail_split(1 if on else 0)
    try:
        yield
    finally:
        lib.gmm_set_tail_split(prev)


def last_path() -> str:
    """Kernel family used by this thread's last launch: "generic", "mfma" or "none"."""
    return {0: "none", _lib.PATH_GENERIC: "generic", _lib.PATH_MFMA: "mfma"}[_lib.load().gmm_last_path()]


def last_kernel() -> str:
    """Kernel of this thread's last launch: "none", "element", "wide", "any" (any alignment, staged through registers),
    "register" or "assembly"."""
    return ("none", "element", "wide", "any", "register", "assembly")[_lib.load().gmm_last_kernel()]
