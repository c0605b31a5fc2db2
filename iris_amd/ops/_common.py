"""Plumbing shared by the operator wrappers: element-type codes, the launch seam, argument checks."""

import logging

import torch

from .. import _lib
from ..host.hip import error_string
from ..host.logging import debug_on, log_rank

_DTYPE_CODES = {
    torch.bfloat16: _lib.BF16,
    torch.float16: _lib.FP16,
    torch.float32: _lib.FP32,
}
_FP8 = getattr(torch, "float8_e4m3fn", None)
if _FP8 is not None:
    _DTYPE_CODES[_FP8] = _lib.FP8_E4M3

_ENTRY_POINTS = {}  # name -> entry point of the kernel library (_lib.launcher())

_PATHS = {"auto": _lib.PATH_AUTO, "mfma": _lib.PATH_MFMA, "generic": _lib.PATH_GENERIC}
_ACC = {"fp32": _lib.ACC_FP32, "reference": _lib.ACC_REFERENCE}


def dtype_code(dtype):
    try:
        return _DTYPE_CODES[dtype]
    except KeyError:
        raise ValueError(f"unsupported dtype {dtype}") from None


def is_fp8(dtype):
    return _FP8 is not None and dtype == _FP8


def path_code(path):
    try:
        return _PATHS[path]
    except KeyError:
        raise ValueError(f"kernel path must be one of {sorted(_PATHS)}, got {path!r}") from None


def acc_code(acc):
    try:
        return _ACC[acc]
    except KeyError:
        raise ValueError(f"slot_sum must be one of {sorted(_ACC)}, got {acc!r}") from None


def require_gpu_tensors(shmem, **tensors):
    """The kernels only run on the GPU that holds the heap."""
    dev = shmem.get_device()
    if dev.type != "cuda":
        raise RuntimeError("fused operators need a GPU context; this Iris context is host-backed")
    for name, t in tensors.items():
        if t is not None and t.device != dev:
            raise RuntimeError(f"{name} is on {t.device}, but the Iris context is on {dev}")


def ptr(t):
    """Device address of a tensor as the entry points take it: a plain integer, None for no tensor."""
    return t.data_ptr() if t is not None else None


def current_stream(shmem):
    """The raw HIP stream torch would launch on for the context's device right now (honours
    `with torch.cuda.stream(...)` and graph capture); None for a host-backed context."""
    device = shmem.get_device_id()
    return torch._C._cuda_getCurrentRawStream(device) if device >= 0 else None


def capturing(stream):
    """True while launches on a raw HIP stream are recorded into a graph."""
    return stream is not None and _lib.library().iris_hip_stream_capturing(stream) != 0


def native(shmem):
    """The module that takes whole operator calls (csrc/launcher.cpp), or None where the Python wrapper has to: on a
    host-backed context and while DEBUG records are wanted.  Its try_<op> functions return None, with nothing done,
    for every call that is not plainly in order - the wrapper then starts over and finds out why - and the entry
    point's result (for check_launch) for the others."""
    return None if shmem.gpu_id < 0 or debug_on() else _lib.launcher()


def rearmed(shmem, workspace, C, operation, shape, dtype, world_size, variant, tiles, stream):
    """True when `workspace` was used by the same call before and needs no preamble to be used again.

    A preamble zeroes flags, aux and C and ends in a barrier, so that no rank's launch meets another rank's
    leftovers.  A process that plays all ranks alone has no such launch beside it: aux, the flags and the
    tiles of C that this rank reduces are overwritten by the launch, the remaining tiles of C are zeroed by the
    launch itself (_lib.CLEAR_C), and work on one stream is ordered without the host waiting for the device
    (decode-sized calls: 32 us with the preamble's three fills and its barrier, 10 us without; 8192 x 4096 reduce-scatter
    150 and 118 us).  Another stream than last time, other shapes or a process group: the preamble runs.  So it does under
    graph capture, which its barrier does not allow, and once a graph holds a launch that uses the buffers: a
    replay does not show here, and may run on any stream.
    """
    if (workspace is None or stream is None or workspace.captured or workspace.stream != stream or workspace.variant != variant or workspace.shape != shape
            or workspace.dtype != dtype or workspace.world_size != world_size or workspace.operation != operation):
        return False
    if variant != "atomic":
        locks, aux = workspace.locks, workspace.aux_buffer
        if locks is None or aux is None or locks.numel() != tiles or aux.shape != C.shape or aux.dtype != C.dtype:
            return False
    return shmem.runs_alone() and not capturing(stream)


def check_launch(err, rank):
    """Raise RuntimeError for an entry point's non-zero result."""
    if err != 0:
        detail = _lib.last_error()
        text = detail if detail else error_string(err)
        log_rank(logging.ERROR, "HIP error code %d: %s", err, text, rank=rank)
        raise RuntimeError(f"HIP error code {err}: {text}")


def iris_launch(entry_name, grid, *args, algorithm, rank, dtype=None):
    """Launch seam: the reference launches `kernel_fn[grid](*args)` here
    (iris/host/tracing/kernel_artifacts.py:54-83); this calls the C entry point of the same operator
    and turns a non-zero hipError_t into RuntimeError the way gpu_try does."""
    if debug_on():
        log_rank(logging.DEBUG, "iris_launch: algorithm=%s kernel=%s grid=%s rank=%d", algorithm, entry_name, grid,
                 rank, rank=rank)
    entry = _ENTRY_POINTS.get(entry_name)
    if entry is None:
        entry = _ENTRY_POINTS[entry_name] = getattr(_lib.launcher(), entry_name)
    check_launch(entry(*args), rank)


def stage_idle_peers(shmem, workspace):
    """One GPU standing in for all ranks: make the other ranks look finished with nothing to add.

    Called by the preambles when the context has `stand_in_peers` set (the benchmark harness sets it):
    the peers' flags are raised and their aux buffers zeroed, so that a fused launch neither waits for
    ranks that do not run nor sums uninitialised memory.  The reference has no counterpart - its peers
    are live processes.
    """
    if not getattr(shmem, "stand_in_peers", False):
        return
    for r in range(shmem.get_num_ranks()):
        if r == shmem.get_rank():
            continue
        if workspace.locks is not None:
            shmem.peer_view(workspace.locks, r).fill_(1)
        if workspace.aux_buffer is not None:
            shmem.peer_view(workspace.aux_buffer, r).zero_()
