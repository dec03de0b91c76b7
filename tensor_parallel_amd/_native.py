"""ctypes binding of `libtpamd.so` (include/tpamd.h).

The library is loaded when this module is imported. If it cannot be loaded, importing still succeeds (so
that rule tables and shape arithmetic can be used on a machine without the build), but every compute
entry point raises `NativeLibraryError`: there is no other implementation to fall back to.
"""
from __future__ import annotations

import ctypes
import functools
import os
from array import array
from pathlib import Path
from typing import Optional, Sequence

import torch  # imported first on purpose: the library binds to the HIP runtime torch has loaded
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

LIB_PATH = Path(__file__).resolve().parent / "_lib" / "libtpamd.so"

EXPORTS = (
    "tpamd_abi_version",
    "tpamd_last_error",
    "tpamd_copy_plan_create",
    "tpamd_copy_plan_run",
    "tpamd_copy_plan_bytes",
    "tpamd_copy_plan_destroy",
    "tpamd_copy_jobs_run",
    "tpamd_transpose_jobs_run",
    "tpamd_scale",
    "tpamd_reduce_partials",
    "tpamd_tuning_reload",
    "tpamd_scratch_query",
    "tpamd_scratch_release",
    "tpamd_linear",
    "tpamd_linear_add",
    "tpamd_linear_noalloc",
    "tpamd_noalloc_scratch_bytes",
    "tpamd_swiglu_up",
    "tpamd_linear_w8",
    "tpamd_attention",
    "tpamd_rms_norm",
    "tpamd_add_rms_norm",
    "tpamd_rope_tables",
    "tpamd_causal_mask",
    "tpamd_rope_append",
    "tpamd_attention_decode_rope",
    "tpamd_attention_decode_rope_devpos",
    "tpamd_linear_ranks",
    "tpamd_swiglu_up_ranks",
    "tpamd_rms_norm_ranks",
    "tpamd_add_rms_norm_ranks",
    "tpamd_attention_decode_rope_ranks",
    "tpamd_linear_w8_ranks",
    "tpamd_linear_add_copy",
    "tpamd_linear_gather_ranks",
    "tpamd_layer_norm_ranks",
    "tpamd_linear_w8_add",
    "tpamd_linear_sum_ranks",
    "tpamd_linear_sum_pays",
    "tpamd_linear_w8_sum_ranks",
    "tpamd_reduce_partials_copy",
    "tpamd_rope",
    "tpamd_rope_tables_ranks",
    "tpamd_causal_mask_ranks",
    "tpamd_add_ranks",
    "tpamd_advance_ranks",
)

ABI_VERSION = 6

BF16, F16, F32 = 0, 1, 2
ACCUM_STEPWISE, ACCUM_F32 = 0, 1
ACT_NONE, ACT_GELU = 0, 1

_DTYPES = {torch.bfloat16: BF16, torch.float16: F16, torch.float32: F32}


class NativeLibraryError(RuntimeError):
    pass


class Unsupported(RuntimeError):
    """The library has no kernel for what it was asked for; nothing was launched."""


class CopyJob(ctypes.Structure):
    _fields_ = [
        ("src", ctypes.c_void_p),
        ("dst", ctypes.c_void_p),
        ("rows", ctypes.c_uint64),
        ("row_bytes", ctypes.c_uint64),
        ("src_pitch", ctypes.c_uint64),
        ("dst_pitch", ctypes.c_uint64),
    ]


class TransposeJob(ctypes.Structure):
    _fields_ = [
        ("src", ctypes.c_void_p),
        ("dst", ctypes.c_void_p),
        ("rows", ctypes.c_uint64),
        ("cols", ctypes.c_uint64),
        ("src_pitch", ctypes.c_uint64),
        ("dst_pitch", ctypes.c_uint64),
    ]


class DecodeRank(ctypes.Structure):
    _fields_ = [(name, ctypes.c_void_p) for name in ("q", "k", "v", "cos", "sin", "k_cache", "v_cache", "out", "pos")]


class W8Rank(ctypes.Structure):
    _fields_ = [(name, ctypes.c_void_p) for name in ("x", "wq", "scale", "outlier_idx", "w_out", "bias", "y")]


_lib: Optional[ctypes.CDLL] = None
_load_error: Optional[str] = None


def _declare(lib: ctypes.CDLL) -> None:
    c = ctypes
    i64, u64, vp, ci = c.c_int64, c.c_uint64, c.c_void_p, c.c_int
    lib.tpamd_abi_version.restype = ci
    lib.tpamd_abi_version.argtypes = []
    lib.tpamd_last_error.restype = c.c_char_p
    lib.tpamd_last_error.argtypes = []
    lib.tpamd_copy_plan_create.restype = ci
    lib.tpamd_copy_plan_create.argtypes = [c.POINTER(CopyJob), c.c_size_t, c.POINTER(vp)]
    lib.tpamd_copy_plan_run.restype = ci
    lib.tpamd_copy_plan_run.argtypes = [vp, vp]
    lib.tpamd_copy_plan_bytes.restype = u64
    lib.tpamd_copy_plan_bytes.argtypes = [vp]
    lib.tpamd_copy_plan_destroy.restype = ci
    lib.tpamd_copy_plan_destroy.argtypes = [vp]
    lib.tpamd_copy_jobs_run.restype = ci
    lib.tpamd_copy_jobs_run.argtypes = [c.POINTER(CopyJob), c.c_size_t, vp]
    lib.tpamd_transpose_jobs_run.restype = ci
    lib.tpamd_transpose_jobs_run.argtypes = [c.POINTER(TransposeJob), c.c_size_t, ci, vp]
    lib.tpamd_scale.restype = ci
    lib.tpamd_scale.argtypes = [vp, vp, u64, ci, ci, ci, vp]
    lib.tpamd_reduce_partials.restype = ci
    lib.tpamd_reduce_partials.argtypes = [c.POINTER(vp), ci, vp, u64, ci, ci, vp]
    lib.tpamd_linear.restype = ci
    lib.tpamd_linear.argtypes = [vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, ci, ci, vp]
    lib.tpamd_linear_add.restype = ci
    lib.tpamd_linear_add.argtypes = [vp, vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, i64, ci, ci, vp]
    lib.tpamd_linear_noalloc.restype = ci
    lib.tpamd_linear_noalloc.argtypes = [vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, ci, ci, vp]
    lib.tpamd_noalloc_scratch_bytes.restype = u64
    lib.tpamd_noalloc_scratch_bytes.argtypes = []
    lib.tpamd_tuning_reload.restype = None
    lib.tpamd_tuning_reload.argtypes = []
    lib.tpamd_scratch_query.restype = ci
    lib.tpamd_scratch_query.argtypes = [vp, c.POINTER(vp), c.POINTER(u64)]
    lib.tpamd_scratch_release.restype = ci
    lib.tpamd_scratch_release.argtypes = [vp]
    lib.tpamd_swiglu_up.restype = ci
    lib.tpamd_swiglu_up.argtypes = [vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, ci, vp]
    lib.tpamd_attention.restype = ci
    lib.tpamd_attention.argtypes = [vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, c.POINTER(i64), c.c_float, ci, ci, vp]
    lib.tpamd_attention_decode_rope.restype = ci
    lib.tpamd_attention_decode_rope.argtypes = [vp, vp, vp, vp, vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, c.POINTER(i64), c.c_float, ci, vp]
    lib.tpamd_attention_decode_rope_devpos.restype = ci
    lib.tpamd_attention_decode_rope_devpos.argtypes = [vp, vp, vp, vp, vp, vp, vp, vp, i64, i64, i64, i64, vp, i64, c.POINTER(i64), c.c_float, ci, vp]
    lib.tpamd_rope_append.restype = ci
    lib.tpamd_rope_append.argtypes = [vp, vp, vp, vp, vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, i64, c.POINTER(i64), ci, vp]
    lib.tpamd_rope.restype = ci
    lib.tpamd_rope.argtypes = [vp, vp, vp, vp, vp, vp, i64, i64, i64, i64, i64, c.POINTER(i64), ci, vp]
    lib.tpamd_rms_norm.restype = ci
    lib.tpamd_rms_norm.argtypes = [vp, vp, vp, i64, i64, i64, i64, c.c_float, ci, vp]
    lib.tpamd_add_rms_norm.restype = ci
    lib.tpamd_add_rms_norm.argtypes = [vp, vp, vp, vp, vp, i64, i64, i64, i64, i64, c.c_float, ci, vp]
    lib.tpamd_rope_tables.restype = ci
    lib.tpamd_rope_tables.argtypes = [vp, ci, vp, i64, i64, i64, i64, i64, c.c_float, vp, vp, ci, vp]
    lib.tpamd_causal_mask.restype = ci
    lib.tpamd_causal_mask.argtypes = [vp, i64, i64, i64, vp, vp]
    pp = vp  # the address of an array of pointers (_Pointers)
    lib.tpamd_linear_ranks.restype = ci
    lib.tpamd_linear_ranks.argtypes = [ci, pp, pp, pp, pp, i64, i64, i64, i64, i64, i64, ci, ci, vp]
    lib.tpamd_linear_gather_ranks.restype = ci
    lib.tpamd_linear_gather_ranks.argtypes = lib.tpamd_linear_ranks.argtypes
    lib.tpamd_linear_add_copy.restype = ci
    lib.tpamd_linear_add_copy.argtypes = [vp, vp, vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, i64, ci, ci, vp]
    lib.tpamd_rope_tables_ranks.restype = ci
    lib.tpamd_rope_tables_ranks.argtypes = [ci, pp, ci, pp, i64, i64, i64, i64, i64, c.c_float, pp, pp, ci, vp]
    lib.tpamd_causal_mask_ranks.restype = ci
    lib.tpamd_causal_mask_ranks.argtypes = [ci, pp, i64, i64, i64, pp, vp]
    lib.tpamd_add_ranks.restype = ci
    lib.tpamd_add_ranks.argtypes = [ci, pp, pp, pp, i64, ci, vp]
    lib.tpamd_advance_ranks.restype = ci
    lib.tpamd_advance_ranks.argtypes = [ci, pp, i64, vp]
    lib.tpamd_swiglu_up_ranks.restype = ci
    lib.tpamd_swiglu_up_ranks.argtypes = [ci, pp, pp, pp, pp, i64, i64, i64, i64, i64, i64, ci, vp]
    lib.tpamd_rms_norm_ranks.restype = ci
    lib.tpamd_rms_norm_ranks.argtypes = [ci, pp, pp, pp, i64, i64, i64, i64, c.c_float, ci, vp]
    lib.tpamd_linear_sum_ranks.restype = ci
    lib.tpamd_linear_sum_ranks.argtypes = [pp, pp, pp, pp, i64, i64, i64, i64, i64, i64, ci, vp]
    lib.tpamd_linear_sum_pays.restype = ci
    lib.tpamd_linear_sum_pays.argtypes = [i64, i64, i64, ci]
    lib.tpamd_linear_w8_sum_ranks.restype = ci
    lib.tpamd_linear_w8_sum_ranks.argtypes = [c.POINTER(W8Rank), i64, i64, i64, i64, i64, i64, i64, i64, ci, vp]
    lib.tpamd_reduce_partials_copy.restype = ci
    lib.tpamd_reduce_partials_copy.argtypes = [pp, ci, vp, vp, u64, ci, ci, vp]
    lib.tpamd_linear_w8_add.restype = ci
    lib.tpamd_linear_w8_add.argtypes = [vp, vp, vp, vp, vp, i64, vp, vp, vp, vp, i64, i64, i64, i64, i64, i64, i64, i64, ci, ci, vp]
    lib.tpamd_layer_norm_ranks.restype = ci
    lib.tpamd_layer_norm_ranks.argtypes = [ci, pp, pp, pp, pp, i64, i64, i64, i64, c.c_float, ci, vp]
    lib.tpamd_add_rms_norm_ranks.restype = ci
    lib.tpamd_add_rms_norm_ranks.argtypes = [ci, pp, pp, pp, pp, pp, i64, i64, i64, i64, i64, c.c_float, ci, vp]
    lib.tpamd_attention_decode_rope_ranks.restype = ci
    lib.tpamd_attention_decode_rope_ranks.argtypes = [ci, c.POINTER(DecodeRank), i64, i64, i64, i64, i64, i64, c.POINTER(i64), c.c_float, ci, vp]
    lib.tpamd_linear_w8_ranks.restype = ci
    lib.tpamd_linear_w8_ranks.argtypes = [ci, c.POINTER(W8Rank), i64, i64, i64, i64, i64, i64, i64, i64, ci, ci, vp]
    lib.tpamd_linear_w8.restype = ci
    lib.tpamd_linear_w8.argtypes = [vp, vp, vp, vp, vp, i64, vp, vp, i64, i64, i64, i64, i64, i64, i64, ci, ci, vp]


def _load() -> None:
    global _lib, _load_error
    path = Path(os.environ.get("TPAMD_LIB", str(LIB_PATH)))
    if not path.exists():
        _load_error = f"{path} does not exist; build it with `python -m tensor_parallel_amd.build`"
        return
    try:
        lib = ctypes.CDLL(str(path))
        for name in EXPORTS:
            getattr(lib, name)
        _declare(lib)
        got = lib.tpamd_abi_version()
        if got != ABI_VERSION:
            raise OSError(f"ABI version {got}, expected {ABI_VERSION}")
        _lib = lib
    except (OSError, AttributeError) as e:  # pragma: no cover - depends on the machine
        _load_error = f"cannot load {path}: {e}"


_load()


def available() -> bool:
    return _lib is not None


def load_error() -> Optional[str]:
    return _load_error


def lib() -> ctypes.CDLL:
    if _lib is None:
        raise NativeLibraryError(f"the HIP library of tensor_parallel_amd is not available: {_load_error}")
    return _lib


def _check(rc: int, what: str) -> None:
    if rc != 0:
        msg = lib().tpamd_last_error().decode("utf-8", "replace")
        if rc == -1:
            raise ValueError(f"{what}: {msg}")
        if rc == -2:
            raise Unsupported(f"{what} failed (status {rc}): {msg}")
        raise RuntimeError(f"{what} failed (status {rc}): {msg}")


def dtype_code(dtype: torch.dtype) -> int:
    try:
        return _DTYPES[dtype]
    except KeyError:
        raise TypeError(f"tensor_parallel_amd kernels support bfloat16, float16 and float32, got {dtype}") from None


def require_device(t: torch.Tensor, what: str) -> None:
    if t.device.type != "cuda":
        raise NativeLibraryError(
            f"{what}: expected a tensor on a HIP device, got {t.device}. tensor_parallel_amd computes on the GPU only."
        )


def on_hip(t: torch.Tensor) -> bool:
    return t.is_cuda


_is_compiling = torch.compiler.is_compiling
_is_tracing = torch._C._is_tracing
_function_modes = torch._C._len_torch_function_stack
_dispatch_modes = torch._C._len_torch_dispatch_stack
_transform = torch._C._functorch.peek_interpreter_stack


def plain_call(*tensors: torch.Tensor) -> bool:
    """Whether a kernel launched on these tensors' memory may stand in for torch calls on them: the tensors are torch's own, and nothing
    follows the calls that would miss the kernel (forward-mode derivatives; vmap and the other functorch transforms, whose wrappers
    have no memory; compilation and tracing; dispatch modes, and function modes other than a default device)."""
    for t in tensors:
        if type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter:
            return False
    if _is_compiling() or _is_tracing() or forward_ad._current_level >= 0 or _transform() is not None or _dispatch_modes():
        return False
    return not _function_modes() or all(type(torch._C._get_function_stack_at(i)) is DeviceContext for i in range(_function_modes()))


def stock_function(f, module: str, qualname: str, names: tuple, variables: tuple) -> bool:
    """Whether f is the function of this name that this module of transformers defines, decorated by nobody but torch and transformers, and known
    here by the names that it looks up and its arguments and locals: a kernel does not stand in for what a program has put in its place."""
    while True:
        if getattr(f, "__code__", None) is None or f.__globals__.get("__name__", "").split(".")[0] not in ("torch", "transformers"):
            return False
        if not hasattr(f, "__wrapped__"):
            break
        f = f.__wrapped__
    return f.__globals__["__name__"] == module and f.__qualname__ == qualname and f.__code__.co_names == names and f.__code__.co_varnames == variables


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def current_stream_ptr(device: torch.device) -> int:
    """Handle of torch's current stream on `device` (the stream every kernel of a call is enqueued on)."""
    if _raw_stream is not None:
        index = device.index
        return _raw_stream(torch.cuda.current_device() if index is None else index)
    return torch.cuda.current_stream(device).cuda_stream


class _on_device:
    """`with _on_device(dev):` makes `dev` the current HIP device for the call; costs nothing when it already is."""

    __slots__ = ("index", "prev")

    def __init__(self, device: torch.device):
        self.index = device.index

    def __enter__(self):
        self.prev = None
        if self.index is not None:
            cur = torch.cuda.current_device()
            if cur != self.index:
                self.prev = cur
                torch.cuda.set_device(self.index)

    def __exit__(self, *exc):
        if self.prev is not None:
            torch.cuda.set_device(self.prev)
        return False


class CopyPlan:
    """A device-resident table of 2-D byte-region copies, run as one kernel launch."""

    def __init__(self, jobs: Sequence[tuple], device: torch.device):
        # jobs: (src_ptr, dst_ptr, rows, row_bytes, src_pitch, dst_pitch)
        self._handle = ctypes.c_void_p()
        self.device = device
        arr = (CopyJob * max(len(jobs), 1))()
        for i, j in enumerate(jobs):
            arr[i] = CopyJob(*j)
        with _on_device(device):
            _check(lib().tpamd_copy_plan_create(arr, len(jobs), ctypes.byref(self._handle)), "tpamd_copy_plan_create")
        self.n_jobs = len(jobs)

    @property
    def nbytes(self) -> int:
        return int(lib().tpamd_copy_plan_bytes(self._handle))

    def run(self, stream_ptr: Optional[int] = None) -> None:
        with _on_device(self.device):
            if stream_ptr is None:
                stream_ptr = current_stream_ptr(self.device)
            _check(lib().tpamd_copy_plan_run(self._handle, ctypes.c_void_p(stream_ptr)), "tpamd_copy_plan_run")

    def close(self) -> None:
        if self._handle:
            h, self._handle = self._handle, ctypes.c_void_p()
            if _lib is not None:
                _lib.tpamd_copy_plan_destroy(h)

    def __del__(self):  # noqa: D105
        try:
            self.close()
        except Exception:
            pass


SMALL_COPY_MAX_JOBS = 16


def run_copy_jobs(jobs: Sequence[tuple], device: torch.device) -> None:
    """Launch up to 16 copy jobs without building a plan (nothing allocated, nothing to keep alive); more jobs go
    through a plan, which is destroyed once its launch has finished."""
    if not jobs:
        return
    with _on_device(device):
        if len(jobs) <= SMALL_COPY_MAX_JOBS:
            arr = (CopyJob * len(jobs))(*[CopyJob(*j) for j in jobs])
            _check(lib().tpamd_copy_jobs_run(arr, len(jobs), ctypes.c_void_p(current_stream_ptr(device))), "tpamd_copy_jobs_run")
            return
    plan = CopyPlan(jobs, device)
    plan.run()
    torch.cuda.current_stream(device).synchronize()  # the plan's tile table must outlive the launch
    plan.close()


TRANSPOSE_MAX_JOBS = 16


def run_transpose_jobs(jobs: Sequence[tuple], elem_bytes: int, device: torch.device) -> None:
    """Launch transposing region moves: jobs are (src_ptr, dst_ptr, rows, cols, src_pitch, dst_pitch) with the extent
    in elements of the source region and the pitches in bytes; 16 jobs per launch."""
    with _on_device(device):
        for at in range(0, len(jobs), TRANSPOSE_MAX_JOBS):
            part = jobs[at:at + TRANSPOSE_MAX_JOBS]
            arr = (TransposeJob * len(part))(*[TransposeJob(*j) for j in part])
            _check(lib().tpamd_transpose_jobs_run(arr, len(part), elem_bytes, ctypes.c_void_p(current_stream_ptr(device))),
                   "tpamd_transpose_jobs_run")


def transpose_regions(src: torch.Tensor, col_ranges: Sequence[tuple], row_range: Optional[tuple] = None,
                      out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """`cat([src[r0:r1, a:b] for a, b in col_ranges], dim=1).t()` as a fresh contiguous tensor, in one launch: column
    ranges (and one row range) are cut out of the row-major 2-D tensor `src` and land transposed, one below the other.
    With the whole tensor as its only range this is `src.t().contiguous()`."""
    require_device(src, "transpose_regions")
    if src.dim() != 2 or src.stride(1) != 1 or src.element_size() not in (1, 2, 4):
        raise ValueError(f"transpose_regions: a row-major 2-D tensor of 1-, 2- or 4-byte elements is needed, got shape {tuple(src.shape)} "
                         f"strides {src.stride()} {src.dtype}")
    r0, r1 = (0, src.shape[0]) if row_range is None else row_range
    if not (0 <= r0 <= r1 <= src.shape[0]) or any(not (0 <= a <= b <= src.shape[1]) for a, b in col_ranges):
        raise ValueError(f"transpose_regions: ranges {row_range} x {list(col_ranges)} outside shape {tuple(src.shape)}")
    es, n_out = src.element_size(), sum(b - a for a, b in col_ranges)
    if out is None:
        out = torch.empty((n_out, r1 - r0), dtype=src.dtype, device=src.device)
    elif out.shape != (n_out, r1 - r0) or out.dtype != src.dtype or out.device != src.device or not out.is_contiguous():
        raise ValueError("transpose_regions: out must be a contiguous tensor of the result's shape, dtype and device")
    pitch, jobs, at = src.stride(0) * es, [], 0
    for a, b in col_ranges:
        if b > a and r1 > r0:
            jobs.append((src.data_ptr() + r0 * pitch + a * es, out.data_ptr() + at * out.stride(0) * es, r1 - r0, b - a, pitch, out.stride(0) * es))
        at += b - a
    run_transpose_jobs(jobs, es, src.device)
    return out


def scale(inp: torch.Tensor, world_size: int, multiply: bool = False) -> torch.Tensor:
    require_device(inp, "scale")
    src = inp.contiguous()
    out = torch.empty_like(src)
    with _on_device(src.device):
        _check(
            lib().tpamd_scale(src.data_ptr(), out.data_ptr(), src.numel(), dtype_code(src.dtype), world_size,
                              1 if multiply else 0, ctypes.c_void_p(current_stream_ptr(src.device))),
            "tpamd_scale",
        )
    return out


def reduce_partials(parts: Sequence[torch.Tensor], accum: int = ACCUM_STEPWISE, out: Optional[torch.Tensor] = None,
                    copy: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The sum of the partials in their order; `copy` (contiguous, as the result) receives it too."""
    if len(parts) == 0:
        raise ValueError("reduce_partials: no partials")
    first = parts[0]
    require_device(first, "reduce_partials")
    keep = []
    for p in parts:
        if p.shape != first.shape or p.dtype != first.dtype or p.device != first.device:
            raise ValueError("reduce_partials: partials must agree in shape, dtype and device")
        keep.append(p.contiguous())
    if out is None:
        out = torch.empty_like(keep[0])
    if copy is not None and (copy.numel() != first.numel() or copy.dtype != first.dtype or copy.device != first.device or not copy.is_contiguous()):
        raise ValueError("reduce_partials: copy must be a contiguous tensor of the result's size, dtype and device")
    ptrs = (ctypes.c_void_p * len(keep))(*[p.data_ptr() for p in keep])
    with _on_device(first.device):
        _check(
            lib().tpamd_reduce_partials_copy(ptrs, len(keep), out.data_ptr(), None if copy is None else copy.data_ptr(), first.numel(),
                                             dtype_code(first.dtype), accum, ctypes.c_void_p(current_stream_ptr(first.device))),
            "tpamd_reduce_partials",
        )
    return out


def _as_2d(x: torch.Tensor) -> torch.Tensor:
    if x.dim() == 2 and x.is_contiguous():
        return x
    x2 = x.reshape(-1, x.shape[-1])
    if x2.stride(-1) != 1 or (x2.shape[0] > 1 and x2.stride(0) < x2.shape[1]):
        x2 = x2.contiguous()
    return x2


def _ld(t: torch.Tensor) -> int:
    return t.stride(0) if t.shape[0] > 1 else max(t.shape[1], 1)


def reload_tuning() -> None:
    """Make the library read its TPAMD_* environment variables again (it reads them once, at load time)."""
    lib().tpamd_tuning_reload()
    _linear_sum_pays.cache_clear()


def scratch_of_stream(device: torch.device, stream_ptr: Optional[int] = None) -> tuple:
    """(address, bytes) of the K-split scratch buffer that work on the stream uses, (None, 0) while it has none."""
    ptr, nbytes = ctypes.c_void_p(), ctypes.c_uint64()
    with _on_device(device):
        if stream_ptr is None:
            stream_ptr = current_stream_ptr(device)
        _check(lib().tpamd_scratch_query(ctypes.c_void_p(stream_ptr), ctypes.byref(ptr), ctypes.byref(nbytes)), "tpamd_scratch_query")
    return ptr.value, int(nbytes.value)


def release_scratch(device: torch.device, stream_ptr: Optional[int] = None) -> None:
    """Free the K-split scratch buffer of a stream that is about to be retired (it is synchronised first)."""
    with _on_device(device):
        if stream_ptr is None:
            stream_ptr = current_stream_ptr(device)
        _check(lib().tpamd_scratch_release(ctypes.c_void_p(stream_ptr)), "tpamd_scratch_release")


def _check_linear(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor]) -> None:
    require_device(x, "linear")
    require_device(w, "linear")
    if x.dtype != w.dtype:
        raise TypeError(f"linear: x is {x.dtype} but w is {w.dtype}")
    if w.dim() != 2 or x.shape[-1] != w.shape[1]:
        raise ValueError(f"linear: x has {x.shape[-1]} input features, w is {tuple(w.shape)}")
    if w.device != x.device:
        raise ValueError(f"linear: x is on {x.device}, w on {w.device}")
    if bias is not None and (bias.shape != (w.shape[0],) or bias.dtype != x.dtype or bias.device != x.device):
        raise ValueError("linear: bias must have shape [N], the dtype of x and live on its device")


# The *_ranks functions take the operands of several ranks whose tensors agree in shape, strides, dtype and device (together.GreenTurn.meet compares
# them): what holds for the first rank's holds for all. They are called once per layer and more of an eager forward, whose pace the host sets.
def _rows(tensors: list) -> tuple:
    """The tensors as row-major matrices with contiguous rows (their memory, where it is one already) and the elements between rows."""
    if tensors[0].is_contiguous():
        return tensors, max(tensors[0].shape[-1], 1)
    tensors = [_as_2d(t) for t in tensors]
    return tensors, _ld(tensors[0])


def _contiguous(tensors: list) -> list:
    return tensors if tensors[0].is_contiguous() else [t.contiguous() for t in tensors]


def _run(what: str, call, index: int, pointers: list, *args) -> None:
    """call(addresses of arrays with the data pointers of each list of tensors (None: no array), *args, stream) on HIP device `index`."""
    n = len(pointers[0])
    block = array("Q", [t.data_ptr() for tensors in pointers if tensors is not None for t in tensors])
    at, where = block.buffer_info()[0], []
    for tensors in pointers:
        where.append(None if tensors is None else at)
        if tensors is not None:
            at += 8 * n
    prev = torch.cuda.current_device()
    if prev != index:
        torch.cuda.set_device(index)
    try:
        rc = call(*where, *args, _raw_stream(index) if _raw_stream is not None else torch.cuda.current_stream(index).cuda_stream)
    finally:
        if prev != index:
            torch.cuda.set_device(prev)
    if rc != 0:
        _check(rc, what)


def _linear_operands(calls: Sequence[tuple]) -> tuple:
    """x, w, bias of all ranks (None: no bias) and the dimensions M, N, K, ldx, ldw."""
    x, w, bias = calls[0]
    _check_linear(x, w, bias)
    N, K = w.shape
    xs, ldx = _rows([c[0] for c in calls])
    ws, ldw = _rows([c[1] for c in calls])
    return xs, ws, None if bias is None else _contiguous([c[2] for c in calls]), (x.numel() // K if K else xs[0].numel(), N, K, ldx, ldw)


def _outputs(x: torch.Tensor, columns: int, n: int) -> list:
    shape = (*x.shape[:-1], columns)
    return [torch.empty(shape, dtype=x.dtype, device=x.device) for _ in range(n)]


def linear_ranks(calls: Sequence[tuple]) -> list:
    """`linear(x, w, bias)` for the (x, w, bias) of several ranks."""
    xs, ws, bs, dims = _linear_operands(calls)
    x, N = calls[0][0], dims[1]
    ys = _outputs(x, N, len(calls))
    _run("tpamd_linear_ranks", functools.partial(lib().tpamd_linear_ranks, len(calls)), x.get_device(), [xs, ws, bs, ys], *dims, N, dtype_code(x.dtype), ACT_NONE)
    return ys


def linear_sum_pays(M: int, N: int, K: int, dtype: torch.dtype, index: Optional[int] = None) -> bool:
    """Whether `linear_sum_ranks` has a launch for these sizes that is faster than two (a rule on sizes, tuning knobs and the CUs of HIP device `index`, of the
    current one if None)."""
    if index is None:
        index = torch.cuda.current_device()
    return index >= 0 and _linear_sum_pays(M, N, K, dtype, index)


@functools.lru_cache(maxsize=4096)
def _linear_sum_pays(M: int, N: int, K: int, dtype: torch.dtype, index: int) -> bool:
    with _on_device(torch.device("cuda", index)):
        return lib().tpamd_linear_sum_pays(M, N, K, dtype_code(dtype)) == 1


def linear_sum_ranks(calls: Sequence[tuple]) -> Optional[list]:
    """The sum of two ranks' `linear(x, w, bias)`, for each a tensor of its own, in one launch; None where there is none for the shape."""
    xs, ws, bs, dims = _linear_operands(calls)
    x, N = calls[0][0], dims[1]
    ys = _outputs(x, N, len(calls))
    try:
        _run("tpamd_linear_sum_ranks", lib().tpamd_linear_sum_ranks, x.get_device(), [xs, ws, bs, ys], *dims, N, dtype_code(x.dtype))
    except Unsupported:
        return None
    return ys


def linear_gather_ranks(calls: Sequence[tuple]) -> list:
    """The `linear(x, w, bias)` of all ranks side by side along the last axis, for each rank a tensor of its own."""
    xs, ws, bs, dims = _linear_operands(calls)
    x, whole = calls[0][0], dims[1] * len(calls)
    ys = _outputs(x, whole, len(calls))
    _run("tpamd_linear_gather_ranks", functools.partial(lib().tpamd_linear_gather_ranks, len(calls)), x.get_device(), [xs, ws, bs, ys], *dims, whole,
         dtype_code(x.dtype), ACT_NONE)
    return ys


def linear(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, act: int = ACT_NONE,
           addend: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None, copy: Optional[torch.Tensor] = None) -> torch.Tensor:
    """y = act(x @ w.T + bias) with w of shape [N, K]; leading dimensions of x are kept. With `addend` (same shape
    and dtype as y): y = (that result, rounded to the dtype) + addend, one step of the sum over rank partials, in the
    same launch. `out` (contiguous, may be `addend`) receives the result; with an addend, `copy` (contiguous) receives it too."""
    _check_linear(x, w, bias)
    N, K = w.shape
    M = x.numel() // K if K else 0
    if addend is not None and (addend.dtype != x.dtype or addend.device != x.device or addend.numel() != M * N
                               or addend.shape[-1] != N):
        raise ValueError("linear: addend must have the shape, dtype and device of the result")
    if out is not None and (out.dtype != x.dtype or out.device != x.device or out.numel() != M * N or not out.is_contiguous()):
        raise ValueError("linear: out must be a contiguous tensor of the result's size, dtype and device")
    if copy is not None and (addend is None or copy.dtype != x.dtype or copy.device != x.device or copy.numel() != M * N or not copy.is_contiguous()):
        raise ValueError("linear: copy goes with an addend and must be a contiguous tensor of the result's size, dtype and device")
    x2, w2 = _as_2d(x), _as_2d(w)
    M = x2.shape[0]
    y = torch.empty((M, N), dtype=x.dtype, device=x.device) if out is None else out.view(M, N)
    b = bias.contiguous() if bias is not None else None
    a2 = _as_2d(addend) if addend is not None else None
    with _on_device(x.device):
        stream = ctypes.c_void_p(current_stream_ptr(x.device))
        if a2 is None:
            _check(
                lib().tpamd_linear(x2.data_ptr(), w2.data_ptr(), b.data_ptr() if b is not None else None, y.data_ptr(),
                                   M, N, K, _ld(x2), _ld(w2), N, dtype_code(x.dtype), act, stream),
                "tpamd_linear",
            )
        elif copy is not None:
            _check(
                lib().tpamd_linear_add_copy(x2.data_ptr(), w2.data_ptr(), b.data_ptr() if b is not None else None, a2.data_ptr(), y.data_ptr(),
                                            copy.data_ptr(), M, N, K, _ld(x2), _ld(w2), _ld(a2), N, dtype_code(x.dtype), act, stream),
                "tpamd_linear_add_copy",
            )
        else:
            _check(
                lib().tpamd_linear_add(x2.data_ptr(), w2.data_ptr(), b.data_ptr() if b is not None else None, a2.data_ptr(),
                                       y.data_ptr(), M, N, K, _ld(x2), _ld(w2), _ld(a2), N, dtype_code(x.dtype), act, stream),
                "tpamd_linear_add",
            )
    return y.view(*x.shape[:-1], N)


def swiglu_up(x: torch.Tensor, wg: torch.Tensor, wu: torch.Tensor) -> torch.Tensor:
    """h = silu(x @ wg.T) * (x @ wu.T)."""
    _check_swiglu_up(x, wg, wu)
    x2, g2, u2 = _as_2d(x), _as_2d(wg), _as_2d(wu)
    if _ld(g2) != _ld(u2):
        u2 = u2.contiguous()
        g2 = g2.contiguous()
    M, K = x2.shape
    N = g2.shape[0]
    h = torch.empty((M, N), dtype=x.dtype, device=x.device)
    with _on_device(x.device):
        _check(
            lib().tpamd_swiglu_up(x2.data_ptr(), g2.data_ptr(), u2.data_ptr(), h.data_ptr(), M, N, K, _ld(x2), _ld(g2), N,
                                  dtype_code(x.dtype), ctypes.c_void_p(current_stream_ptr(x.device))),
            "tpamd_swiglu_up",
        )
    return h.view(*x.shape[:-1], N)


def _check_swiglu_up(x: torch.Tensor, wg: torch.Tensor, wu: torch.Tensor) -> None:
    require_device(x, "swiglu_up")
    if not (x.dtype == wg.dtype == wu.dtype):
        raise TypeError("swiglu_up: x, wg, wu must share one dtype")
    if wg.dim() != 2 or wg.shape != wu.shape or x.shape[-1] != wg.shape[1]:
        raise ValueError("swiglu_up: shape mismatch")
    if wg.device != x.device or wu.device != x.device:
        raise ValueError(f"swiglu_up: x is on {x.device}, wg on {wg.device}, wu on {wu.device}")


def swiglu_up_ranks(calls: Sequence[tuple]) -> list:
    """`swiglu_up(x, wg, wu)` for the operands of several ranks."""
    x, wg, wu = calls[0]
    _check_swiglu_up(x, wg, wu)
    xs, ldx = _rows([c[0] for c in calls])
    gs, ldg = _rows([c[1] for c in calls])
    us, ldu = _rows([c[2] for c in calls])
    N, K = wg.shape
    if ldg != ldu:
        gs, us, ldg = [g.contiguous() for g in gs], [u.contiguous() for u in us], max(K, 1)
    hs = _outputs(x, N, len(calls))
    _run("tpamd_swiglu_up_ranks", functools.partial(lib().tpamd_swiglu_up_ranks, len(calls)), x.get_device(), [xs, gs, us, hs],
         x.numel() // K if K else xs[0].numel(), N, K, ldx, ldg, N, dtype_code(x.dtype))
    return hs


def rms_norm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """w * (x * rsqrt(mean(x^2) + eps)) over the last axis, sums in fp32, rounded as the two products of tensors of x's dtype."""
    return rms_norm_ranks([(x, w, eps)])[0]


def rms_norm_ranks(calls: Sequence[tuple]) -> list:
    """`rms_norm(x, w, eps)` for the operands of several ranks (with one eps)."""
    x, w, eps = calls[0]
    require_device(x, "rms_norm")
    if w.dtype != x.dtype or w.get_device() != x.get_device() or w.dim() != 1 or x.dim() == 0 or x.shape[-1] != w.shape[0]:
        raise ValueError(f"rms_norm: x {tuple(x.shape)} {x.dtype} on {x.device} and w {tuple(w.shape)} {w.dtype} on {w.device} do not fit")
    D = w.shape[0]
    xs, ldx = _rows([c[0] for c in calls])
    ys = _outputs(x, D, len(calls))
    if D:
        _run("tpamd_rms_norm", functools.partial(lib().tpamd_rms_norm_ranks, len(calls)), x.get_device(), [xs, _contiguous([c[1] for c in calls]), ys],
             x.numel() // D, D, ldx, D, float(eps), dtype_code(x.dtype))
    return ys


def add_rms_norm(r: torch.Tensor, x: torch.Tensor, w: torch.Tensor, eps: float) -> tuple:
    """(r + x, the RMS norm of that sum) of two tensors of one shape, dtype and device; arithmetic as in `rms_norm`."""
    return add_rms_norm_ranks([(r, x, w, eps)])[0]


def add_rms_norm_ranks(calls: Sequence[tuple]) -> list:
    """`add_rms_norm(r, x, w, eps)` for the operands of several ranks (with one eps)."""
    r, x, w, eps = calls[0]
    require_device(x, "add_rms_norm")
    if (r.shape != x.shape or r.dtype != x.dtype or r.get_device() != x.get_device() or w.dtype != x.dtype or w.get_device() != x.get_device() or w.dim() != 1
            or x.dim() == 0 or x.shape[-1] != w.shape[0]):
        raise ValueError(f"add_rms_norm: r {tuple(r.shape)} {r.dtype} on {r.device}, x {tuple(x.shape)} {x.dtype} on {x.device} and w {tuple(w.shape)} "
                         f"{w.dtype} on {w.device} do not fit")
    D = w.shape[0]
    xs, ldx = _rows([c[1] for c in calls])
    rs, ldr = _rows([c[0] for c in calls])
    totals, ys = _outputs(x, D, len(calls)), _outputs(x, D, len(calls))
    if D:
        _run("tpamd_add_rms_norm", functools.partial(lib().tpamd_add_rms_norm_ranks, len(calls)), x.get_device(),
             [xs, rs, _contiguous([c[2] for c in calls]), totals, ys], x.numel() // D, D, ldx, ldr, D, float(eps), dtype_code(x.dtype))
    return list(zip(totals, ys))


def layer_norm(x: torch.Tensor, w: torch.Tensor, b: Optional[torch.Tensor], eps: float) -> torch.Tensor:
    """(x - mean) * rsqrt(var + eps) * w + b over the last axis, in fp32, rounded once."""
    return layer_norm_ranks([(x, w, b, eps)])[0]


def layer_norm_ranks(calls: Sequence[tuple]) -> list:
    """`layer_norm(x, w, b, eps)` for the operands of several ranks (with one eps)."""
    x, w, b, eps = calls[0]
    require_device(x, "layer_norm")
    for t in (w, b):
        if t is not None and (t.dtype != x.dtype or t.get_device() != x.get_device() or t.dim() != 1 or x.dim() == 0 or x.shape[-1] != t.shape[0]):
            raise ValueError(f"layer_norm: x {tuple(x.shape)} {x.dtype} on {x.device} and {tuple(t.shape)} {t.dtype} on {t.device} do not fit")
    D = w.shape[0]
    xs, ldx = _rows([c[0] for c in calls])
    ys = _outputs(x, D, len(calls))
    if D:
        _run("tpamd_layer_norm", functools.partial(lib().tpamd_layer_norm_ranks, len(calls)), x.get_device(),
             [xs, _contiguous([c[1] for c in calls]), None if b is None else _contiguous([c[2] for c in calls]), ys], x.numel() // D, D, ldx, D, float(eps),
             dtype_code(x.dtype))
    return ys


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: Optional[float] = None, causal: bool = True,
              out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """softmax(scale * q k^T [+ causal]) v. q [B, Hq, Sq, D], k / v [B, Hkv, Skv, D] -> [B, Sq, Hq, D] (the layout the
    attention output projection consumes). Grouped-query heads when Hq > Hkv; causal is aligned to the END of the key
    range (query i sees keys j <= i + Skv - Sq). `out`, if given, is a [B, Sq, Hq, D] tensor (or view) of q's dtype and
    device whose rows are contiguous and start on 8-byte boundaries."""
    require_device(q, "attention")
    if not (q.dtype == k.dtype == v.dtype) or q.dtype not in (torch.bfloat16, torch.float16):
        raise TypeError("attention: q, k, v must share bfloat16 or float16")
    if q.dim() != 4 or k.dim() != 4 or v.shape != k.shape or q.shape[0] != k.shape[0] or q.shape[3] != k.shape[3]:
        raise ValueError(f"attention: shapes q {tuple(q.shape)}, k {tuple(k.shape)}, v {tuple(v.shape)} do not fit")
    if k.device != q.device or v.device != q.device:
        raise ValueError(f"attention: q is on {q.device}, k on {k.device}, v on {v.device}")
    B, Hq, Sq, D = q.shape
    Hkv, Skv = k.shape[1], k.shape[2]
    q, k, v = (t if t.stride(3) == 1 else t.contiguous() for t in (q, k, v))
    if out is None:
        out = torch.empty((B, Sq, Hq, D), dtype=q.dtype, device=q.device)
    elif out.shape != (B, Sq, Hq, D) or out.dtype != q.dtype or out.device != q.device or out.stride(3) != 1:
        raise ValueError(f"attention: out must be a [{B}, {Sq}, {Hq}, {D}] {q.dtype} tensor on {q.device} with contiguous rows")
    strides = (ctypes.c_int64 * 12)(q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
                                    v.stride(0), v.stride(1), v.stride(2), out.stride(0), out.stride(1), out.stride(2))
    with _on_device(q.device):
        _check(
            lib().tpamd_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), B, Hq, Hkv, Sq, Skv, D, strides,
                                  float(scale if scale is not None else D ** -0.5), 1 if causal else 0, dtype_code(q.dtype),
                                  ctypes.c_void_p(current_stream_ptr(q.device))),
            "tpamd_attention",
        )
    return out


def rope_tables(inv_freq: torch.Tensor, position_ids: torch.Tensor, scaling: float, dtype: torch.dtype) -> tuple:
    """(cos, sin) [B, S, 2 * len(inv_freq)] of the angles position * inv_freq, scaled, in `dtype` (arithmetic in fp32)."""
    require_device(position_ids, "rope_tables")
    if inv_freq.dim() != 1 or position_ids.dim() != 2 or position_ids.dtype != torch.int64 or inv_freq.device != position_ids.device:
        raise ValueError(f"rope_tables: inv_freq {tuple(inv_freq.shape)} and int64 position_ids [B, S] on one device are needed, got "
                         f"{tuple(position_ids.shape)} {position_ids.dtype}")
    B, S = position_ids.shape
    half = inv_freq.shape[0]
    inv_freq = inv_freq.contiguous()
    cos = torch.empty((B, S, 2 * half), dtype=dtype, device=position_ids.device)
    sin = torch.empty_like(cos)
    with _on_device(position_ids.device):
        _check(
            lib().tpamd_rope_tables(inv_freq.data_ptr(), dtype_code(inv_freq.dtype), position_ids.data_ptr(), position_ids.stride(0),
                                    position_ids.stride(1), B, S, half, float(scaling), cos.data_ptr(), sin.data_ptr(), dtype_code(dtype),
                                    ctypes.c_void_p(current_stream_ptr(position_ids.device))),
            "tpamd_rope_tables",
        )
    return cos, sin


def causal_mask(q_offset: torch.Tensor, kv_offset: int, q_length: int, kv_length: int) -> torch.Tensor:
    """Boolean [1, 1, q_length, kv_length]: kv_offset + j <= q_offset + i, the offset of the queries (one int64) read on the device."""
    require_device(q_offset, "causal_mask")
    if q_offset.dtype != torch.int64 or q_offset.numel() != 1:
        raise ValueError(f"causal_mask: q_offset must be one int64, got {tuple(q_offset.shape)} {q_offset.dtype}")
    out = torch.empty((1, 1, q_length, kv_length), dtype=torch.bool, device=q_offset.device)
    with _on_device(q_offset.device):
        _check(
            lib().tpamd_causal_mask(q_offset.data_ptr(), kv_offset, q_length, kv_length, out.data_ptr(),
                                    ctypes.c_void_p(current_stream_ptr(q_offset.device))),
            "tpamd_causal_mask",
        )
    return out


def rope_tables_ranks(calls: Sequence[tuple]) -> list:
    """`rope_tables(inv_freq, position_ids, scaling, dtype)` for the operands of several ranks (with one scaling and dtype)."""
    inv_freq, position_ids, scaling, dtype = calls[0]
    require_device(position_ids, "rope_tables")
    if inv_freq.dim() != 1 or position_ids.dim() != 2 or position_ids.dtype != torch.int64 or inv_freq.device != position_ids.device:
        raise ValueError(f"rope_tables: inv_freq {tuple(inv_freq.shape)} and int64 position_ids [B, S] on one device are needed, got "
                         f"{tuple(position_ids.shape)} {position_ids.dtype}")
    B, S = position_ids.shape
    half = inv_freq.shape[0]
    cos = [torch.empty((B, S, 2 * half), dtype=dtype, device=position_ids.device) for _ in calls]
    sin = [torch.empty_like(c) for c in cos]
    n, table = len(calls), lib().tpamd_rope_tables_ranks
    code, pos_b, pos_s = dtype_code(inv_freq.dtype), position_ids.stride(0), position_ids.stride(1)
    _run("tpamd_rope_tables", lambda f, p, c, s, stream: table(n, f, code, p, pos_b, pos_s, B, S, half, float(scaling), c, s, dtype_code(dtype), stream),
         position_ids.get_device(), [_contiguous([c[0] for c in calls]), [c[1] for c in calls], cos, sin])
    return list(zip(cos, sin))


def causal_mask_ranks(calls: Sequence[tuple]) -> list:
    """`causal_mask(q_offset, kv_offset, q_length, kv_length)` for the offsets of several ranks (with the same numbers)."""
    q_offset, kv_offset, q_length, kv_length = calls[0]
    require_device(q_offset, "causal_mask")
    if q_offset.dtype != torch.int64 or q_offset.numel() != 1:
        raise ValueError(f"causal_mask: q_offset must be one int64, got {tuple(q_offset.shape)} {q_offset.dtype}")
    masks = [torch.empty((1, 1, q_length, kv_length), dtype=torch.bool, device=q_offset.device) for _ in calls]
    n, mask = len(calls), lib().tpamd_causal_mask_ranks
    _run("tpamd_causal_mask", lambda q, out, stream: mask(n, q, kv_offset, q_length, kv_length, out, stream), q_offset.get_device(), [[c[0] for c in calls], masks])
    return masks


def add_ranks(calls: Sequence[tuple]) -> list:
    """a + b of several ranks, tensors of one shape and dtype."""
    a, b = calls[0]
    require_device(a, "add_ranks")
    if a.shape != b.shape or a.dtype != b.dtype or a.get_device() != b.get_device():
        raise ValueError(f"add_ranks: {tuple(a.shape)} {a.dtype} and {tuple(b.shape)} {b.dtype} do not fit")
    xs, rs = _contiguous([c[0] for c in calls]), _contiguous([c[1] for c in calls])
    if any(t.data_ptr() % 16 for t in xs + rs):
        return [x + r for x, r in calls]
    outs = [torch.empty_like(x) for x in xs]
    _run("tpamd_add_ranks", functools.partial(lib().tpamd_add_ranks, len(calls)), a.get_device(), [xs, rs, outs], a.numel(), dtype_code(a.dtype))
    return outs


def advance_ranks(calls: Sequence[tuple]) -> list:
    """count.add_(by) for the int64 counts of several ranks."""
    count, by = calls[0]
    require_device(count, "advance_ranks")
    if count.dtype != torch.int64 or count.numel() != 1:
        raise ValueError(f"advance_ranks: a count must be one int64, got {tuple(count.shape)} {count.dtype}")
    if len({c.data_ptr() for c, _ in calls}) < len(calls):  # ranks that share a count: one after the other
        return [c.add_(by) for c, by in calls]
    _run("tpamd_advance_ranks", functools.partial(lib().tpamd_advance_ranks, len(calls)), count.get_device(), [[c[0] for c in calls]], by)
    return [c[0] for c in calls]


def rope_append(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                k_cache: torch.Tensor, v_cache: torch.Tensor, pos0: int, q_out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Rotary embedding of the new rows and their hand-over to the rank-local cache, one launch.
    q [B, S, Hq, D] or [B, S, Hkv, Hq / Hkv, D] (the query heads of each key/value head, as a fused projection that
    interleaves them with their key and value lays them out), k / v [B, S, Hkv, D] (all views of a projection output),
    cos / sin [B or 1, S, D];
    k_cache / v_cache [B, Hkv, L, D] are written in place at positions pos0 .. pos0 + S - 1 (rotated k, v);
    returns the rotated q as [B, Hq, S, D], the layout `attention` takes."""
    require_device(q, "rope_append")
    if not (q.dtype == k.dtype == v.dtype == cos.dtype == sin.dtype == k_cache.dtype == v_cache.dtype) or q.dtype not in (
            torch.bfloat16, torch.float16):
        raise TypeError("rope_append: every tensor must share bfloat16 or float16")
    if q.dim() not in (4, 5) or k.dim() != 4 or v.shape != k.shape or q.shape[:2] != k.shape[:2] or q.shape[-1] != k.shape[3] or (
            q.dim() == 5 and q.shape[2] != k.shape[2]):
        raise ValueError(f"rope_append: shapes q {tuple(q.shape)}, k {tuple(k.shape)}, v {tuple(v.shape)} do not fit")
    B, S, Hkv, D = k.shape
    Hq = q.shape[2] if q.dim() == 4 else q.shape[2] * q.shape[3]
    if Hq % Hkv:
        raise ValueError(f"rope_append: {Hq} query heads over {Hkv} key/value heads")
    q_head, q_group = (q.stride(2), q.stride(2) * (Hq // Hkv)) if q.dim() == 4 else (q.stride(3), q.stride(2))
    if cos.dim() == 2:
        cos, sin = cos.unsqueeze(0), sin.unsqueeze(0)
    if cos.shape != sin.shape or cos.dim() != 3 or cos.shape[0] not in (1, B) or cos.shape[1:] != (S, D):
        raise ValueError(f"rope_append: cos / sin must be [{B} or 1, {S}, {D}], got {tuple(cos.shape)} / {tuple(sin.shape)}")
    if k_cache.dim() != 4 or v_cache.shape != k_cache.shape or k_cache.shape[0] != B or k_cache.shape[1] != Hkv or k_cache.shape[3] != D:
        raise ValueError(f"rope_append: caches must be [{B}, {Hkv}, L, {D}], got {tuple(k_cache.shape)} / {tuple(v_cache.shape)}")
    for name, t in (("k", k), ("v", v), ("cos", cos), ("sin", sin), ("k_cache", k_cache), ("v_cache", v_cache)):
        if t.device != q.device:
            raise ValueError(f"rope_append: q is on {q.device}, {name} on {t.device}")
        if t.stride(-1) != 1:
            raise ValueError(f"rope_append: {name} must have contiguous rows")
    if q.stride(-1) != 1:
        raise ValueError("rope_append: q must have contiguous rows")
    if sin.stride() != cos.stride():
        sin = sin.contiguous()
        cos = cos.contiguous()
    if q_out is None:
        q_out = torch.empty((B, Hq, S, D), dtype=q.dtype, device=q.device)
    elif q_out.shape != (B, Hq, S, D) or q_out.dtype != q.dtype or q_out.device != q.device or q_out.stride(3) != 1:
        raise ValueError(f"rope_append: q_out must be a [{B}, {Hq}, {S}, {D}] {q.dtype} tensor on {q.device} with contiguous rows")
    strides = (ctypes.c_int64 * 21)(q.stride(0), q.stride(1), q_head, k.stride(0), k.stride(1), k.stride(2),
                                    v.stride(0), v.stride(1), v.stride(2), cos.stride(0) if cos.shape[0] > 1 else 0, cos.stride(1),
                                    q_out.stride(0), q_out.stride(1), q_out.stride(2), k_cache.stride(0), k_cache.stride(1),
                                    k_cache.stride(2), v_cache.stride(0), v_cache.stride(1), v_cache.stride(2), q_group)
    with _on_device(q.device):
        _check(
            lib().tpamd_rope_append(q.data_ptr(), k.data_ptr(), v.data_ptr(), cos.data_ptr(), sin.data_ptr(), q_out.data_ptr(),
                                    k_cache.data_ptr(), v_cache.data_ptr(), B, S, Hq, Hkv, D, int(pos0), k_cache.shape[2], strides,
                                    dtype_code(q.dtype), ctypes.c_void_p(current_stream_ptr(q.device))),
            "tpamd_rope_append",
        )
    return q_out


def _decode_operands(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, k_cache: torch.Tensor,
                     v_cache: torch.Tensor) -> tuple:
    """Checks the operands of a decode step; (elements between query heads, between groups of them, cos, sin as rows of D)."""
    require_device(q, "attention_decode_rope")
    if not (q.dtype == k.dtype == v.dtype == cos.dtype == sin.dtype == k_cache.dtype == v_cache.dtype) or q.dtype not in (
            torch.bfloat16, torch.float16):
        raise TypeError("attention_decode_rope: every tensor must share bfloat16 or float16")
    if q.dim() not in (4, 5) or k.dim() != 4 or v.shape != k.shape or q.shape[:2] != k.shape[:2] or k.shape[1] != 1 or \
            q.shape[-1] != k.shape[3] or (q.dim() == 5 and q.shape[2] != k.shape[2]):
        raise ValueError(f"attention_decode_rope: shapes q {tuple(q.shape)}, k {tuple(k.shape)}, v {tuple(v.shape)} do not fit one new position")
    B, _, Hkv, D = k.shape
    Hq = q.shape[2] if q.dim() == 4 else q.shape[2] * q.shape[3]
    if Hq % Hkv:
        raise ValueError(f"attention_decode_rope: {Hq} query heads over {Hkv} key/value heads")
    q_head, q_group = (q.stride(2), q.stride(2) * (Hq // Hkv)) if q.dim() == 4 else (q.stride(3), q.stride(2))
    cos, sin = cos.reshape(-1, D), sin.reshape(-1, D)
    if cos.shape != sin.shape or cos.shape[0] not in (1, B):
        raise ValueError(f"attention_decode_rope: cos / sin must hold [{B} or 1] rows of {D}, got {tuple(cos.shape)} / {tuple(sin.shape)}")
    if k_cache.dim() != 4 or v_cache.shape != k_cache.shape or k_cache.shape[0] != B or k_cache.shape[1] != Hkv or k_cache.shape[3] != D:
        raise ValueError(f"attention_decode_rope: caches must be [{B}, {Hkv}, L, {D}], got {tuple(k_cache.shape)} / {tuple(v_cache.shape)}")
    for name, t in (("q", q), ("k", k), ("v", v), ("cos", cos), ("sin", sin), ("k_cache", k_cache), ("v_cache", v_cache)):
        if t.device != q.device:
            raise ValueError(f"attention_decode_rope: q is on {q.device}, {name} on {t.device}")
        if t.stride(-1) != 1:
            raise ValueError(f"attention_decode_rope: {name} must have contiguous rows")
    if sin.stride() != cos.stride():
        sin, cos = sin.contiguous(), cos.contiguous()
    return q_head, q_group, cos, sin


def _decode_strides(q, q_head: int, q_group: int, k, v, cos, k_cache, v_cache, out):
    return (ctypes.c_int64 * 16)(q.stride(0), q_head, q_group, k.stride(0), k.stride(2), v.stride(0), v.stride(2),
                                 cos.stride(0) if cos.shape[0] > 1 else 0, k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
                                 v_cache.stride(0), v_cache.stride(1), v_cache.stride(2), out.stride(0), out.stride(2))


def _check_device_position(q: torch.Tensor, pos0: torch.Tensor) -> None:
    if pos0.dtype != torch.int64 or pos0.numel() != 1 or pos0.device != q.device:
        raise ValueError(f"attention_decode_rope: a position on the device must be one int64 element on {q.device}, "
                         f"got {tuple(pos0.shape)} {pos0.dtype} on {pos0.device}")


def attention_decode_rope_ranks(calls: Sequence[tuple]) -> list:
    """`attention_decode_rope(q, k, v, cos, sin, k_cache, v_cache, pos0, scale)` for the operands of several ranks (with one scale, and one pos0
    where that is a number)."""
    q, k, v, cos, sin, k_cache, v_cache, pos0, scale = calls[0]
    q_head, q_group, cos, sin = _decode_operands(q, k, v, cos, sin, k_cache, v_cache)
    on_device = isinstance(pos0, torch.Tensor)
    if on_device:
        _check_device_position(q, pos0)
    B, _, Hkv, D = k.shape
    Hq = q.shape[2] if q.dim() == 4 else q.shape[2] * q.shape[3]
    ranks, keep = (DecodeRank * len(calls))(), []
    for rank, (rq, rk, rv, rcos, rsin, rk_cache, rv_cache, rpos, _) in zip(ranks, calls):
        rcos, rsin = rcos.reshape(-1, D), rsin.reshape(-1, D)
        if rsin.stride() != rcos.stride():
            rsin, rcos = rsin.contiguous(), rcos.contiguous()
        out = torch.empty((B, 1, Hq, D), dtype=q.dtype, device=q.device)
        keep.append((rcos, rsin, out))
        rank.q, rank.k, rank.v, rank.cos, rank.sin = rq.data_ptr(), rk.data_ptr(), rv.data_ptr(), rcos.data_ptr(), rsin.data_ptr()
        rank.k_cache, rank.v_cache, rank.out, rank.pos = rk_cache.data_ptr(), rv_cache.data_ptr(), out.data_ptr(), rpos.data_ptr() if on_device else None
    strides = _decode_strides(q, q_head, q_group, k, v, cos, k_cache, v_cache, out)
    with _on_device(q.device):
        rc = lib().tpamd_attention_decode_rope_ranks(len(calls), ranks, B, Hq, Hkv, D, 0 if on_device else int(pos0), k_cache.shape[2], strides,
                                                     float(scale if scale is not None else D ** -0.5), dtype_code(q.dtype),
                                                     ctypes.c_void_p(current_stream_ptr(q.device)))
    if rc == -2 and not on_device:  # no scratch buffer for this stream: rank by rank, with the two calls that need none
        return [attention_decode_rope(*call) for call in calls]
    _check(rc, "tpamd_attention_decode_rope_ranks")
    return [out for _, _, out in keep]


def rope_takes(B: int, S: int, heads: int, D: int) -> bool:
    """Whether `rope` rotates `heads` query and key heads of this many sequences and positions in a launch (which has fewer than 2^32 threads)."""
    return B < 1 << 24 and S < 1 << 24 and heads < 1 << 16 and B * S * ((heads * (D // 16) + 255) // 256) < 1 << 24


def rope(q: torch.Tensor, k: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> tuple:
    """Rotary embedding of whole sequences in one launch: q [B, S, Hq, D], k [B, S, Hkv, D] (views of projection outputs), cos / sin [B or 1, S, D];
    returns them rotated, as [B, Hq, S, D] and [B, Hkv, S, D]. Arithmetic as in `rope_append`."""
    require_device(q, "rope")
    if not (q.dtype == k.dtype == cos.dtype == sin.dtype) or q.dtype not in (torch.bfloat16, torch.float16):
        raise TypeError("rope: every tensor must share bfloat16 or float16")
    B, S, Hq, D = q.shape
    if k.dim() != 4 or k.shape[:2] != (B, S) or k.shape[3] != D or cos.shape != sin.shape or cos.dim() != 3 or cos.shape[0] not in (1, B) or cos.shape[1:] != (S, D):
        raise ValueError(f"rope: shapes q {tuple(q.shape)}, k {tuple(k.shape)}, cos {tuple(cos.shape)}, sin {tuple(sin.shape)} do not fit")
    for name, t in (("q", q), ("k", k), ("cos", cos), ("sin", sin)):
        if t.device != q.device or t.stride(-1) != 1:
            raise ValueError(f"rope: {name} must have contiguous rows on {q.device}")
    if sin.stride() != cos.stride():
        sin, cos = sin.contiguous(), cos.contiguous()
    Hkv = k.shape[2]
    q_out = torch.empty((B, Hq, S, D), dtype=q.dtype, device=q.device)
    k_out = torch.empty((B, Hkv, S, D), dtype=q.dtype, device=q.device)
    strides = (ctypes.c_int64 * 14)(*q.stride()[:3], *k.stride()[:3], cos.stride(0) if cos.shape[0] > 1 else 0, cos.stride(1), *q_out.stride()[:3], *k_out.stride()[:3])
    with _on_device(q.device):
        _check(
            lib().tpamd_rope(q.data_ptr(), k.data_ptr(), cos.data_ptr(), sin.data_ptr(), q_out.data_ptr(), k_out.data_ptr(), B, S, Hq, Hkv, D, strides,
                             dtype_code(q.dtype), ctypes.c_void_p(current_stream_ptr(q.device))),
            "tpamd_rope",
        )
    return q_out, k_out


def attention_decode_rope(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                          k_cache: torch.Tensor, v_cache: torch.Tensor, pos0, scale: Optional[float] = None,
                          out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """`rope_append` and `attention` for one new position per sequence, in one or two launches instead of two or three.
    q [B, 1, Hq, D] or [B, 1, Hkv, Hq / Hkv, D], k / v [B, 1, Hkv, D] (views of the projection output), cos / sin [B or 1, 1, D]
    (or [1, D] / [D]); the caches [B, Hkv, L, D] hold pos0 positions and receive the new one at pos0. Returns [B, 1, Hq, D].
    Where the library has no scratch buffer for the stream (first use under graph capture) the two calls are made instead.

    `pos0` may also be an int64 tensor of one element on the device: the kernels then read the count when they run
    (`tpamd_attention_decode_rope_devpos`), the launches are laid out for the L positions the caches can hold, and the call
    can sit in a HIP graph that is replayed for every decode step. The caller advances the count."""
    q_head, q_group, cos, sin = _decode_operands(q, k, v, cos, sin, k_cache, v_cache)
    B, _, Hkv, D = k.shape
    Hq = q.shape[2] if q.dim() == 4 else q.shape[2] * q.shape[3]
    if out is None:
        out = torch.empty((B, 1, Hq, D), dtype=q.dtype, device=q.device)
    elif out.shape != (B, 1, Hq, D) or out.dtype != q.dtype or out.device != q.device or out.stride(3) != 1:
        raise ValueError(f"attention_decode_rope: out must be a [{B}, 1, {Hq}, {D}] {q.dtype} tensor on {q.device} with contiguous rows")
    strides = _decode_strides(q, q_head, q_group, k, v, cos, k_cache, v_cache, out)
    if isinstance(pos0, torch.Tensor):
        _check_device_position(q, pos0)
        with _on_device(q.device):
            rc = lib().tpamd_attention_decode_rope_devpos(q.data_ptr(), k.data_ptr(), v.data_ptr(), cos.data_ptr(), sin.data_ptr(),
                                                          k_cache.data_ptr(), v_cache.data_ptr(), out.data_ptr(), B, Hq, Hkv, D,
                                                          ctypes.c_void_p(pos0.data_ptr()), k_cache.shape[2], strides,
                                                          float(scale if scale is not None else D ** -0.5), dtype_code(q.dtype),
                                                          ctypes.c_void_p(current_stream_ptr(q.device)))
        _check(rc, "tpamd_attention_decode_rope_devpos")
        return out
    with _on_device(q.device):
        rc = lib().tpamd_attention_decode_rope(q.data_ptr(), k.data_ptr(), v.data_ptr(), cos.data_ptr(), sin.data_ptr(),
                                               k_cache.data_ptr(), v_cache.data_ptr(), out.data_ptr(), B, Hq, Hkv, D, int(pos0),
                                               k_cache.shape[2], strides, float(scale if scale is not None else D ** -0.5),
                                               dtype_code(q.dtype), ctypes.c_void_p(current_stream_ptr(q.device)))
    if rc == -2 and B > 0 and D in (64, 128):  # no scratch buffer for this stream: the two-call sequence needs none
        q_rot = rope_append(q, k, v, cos.unsqueeze(1), sin.unsqueeze(1), k_cache, v_cache, pos0)
        return attention(q_rot, k_cache[:, :, :pos0 + 1], v_cache[:, :, :pos0 + 1], scale=scale, causal=True, out=out)
    _check(rc, "tpamd_attention_decode_rope")
    return out


def linear_w8(x: torch.Tensor, wq: torch.Tensor, scale_: torch.Tensor, outlier_idx: Optional[torch.Tensor],
              w_out: Optional[torch.Tensor], bias: Optional[torch.Tensor] = None, act: int = ACT_NONE,
              addend: Optional[torch.Tensor] = None, copy: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Weight-only int8 Linear with outlier columns kept in the activation dtype. `addend` and `copy` as in `linear`."""
    (x2, wq, scale_, outlier_idx, w_out, b), (M, N, K, n_out) = _w8_operands(x, wq, scale_, outlier_idx, w_out, bias)
    if addend is not None and (addend.dtype != x.dtype or addend.device != x.device or addend.numel() != M * N or addend.shape[-1] != N):
        raise ValueError("linear_w8: addend must have the shape, dtype and device of the result")
    if copy is not None and (addend is None or copy.dtype != x.dtype or copy.device != x.device or copy.numel() != M * N or not copy.is_contiguous()):
        raise ValueError("linear_w8: copy goes with an addend and must be a contiguous tensor of the result's size, dtype and device")
    y = torch.empty((M, N), dtype=x.dtype, device=x.device)
    head = (x2.data_ptr(), wq.data_ptr(), scale_.data_ptr(), outlier_idx.data_ptr() if n_out else None, w_out.data_ptr() if n_out else None, n_out,
            b.data_ptr() if b is not None else None)
    with _on_device(x.device):
        stream = ctypes.c_void_p(current_stream_ptr(x.device))
        if addend is None:
            _check(
                lib().tpamd_linear_w8(*head, y.data_ptr(), M, N, K, _ld(x2), K, max(n_out, 1), N, dtype_code(x.dtype), act, stream),
                "tpamd_linear_w8",
            )
        else:
            a2 = _as_2d(addend)
            _check(
                lib().tpamd_linear_w8_add(*head, a2.data_ptr(), y.data_ptr(), None if copy is None else copy.data_ptr(), M, N, K, _ld(x2), K, max(n_out, 1),
                                          _ld(a2), N, dtype_code(x.dtype), act, stream),
                "tpamd_linear_w8_add",
            )
    return y.view(*x.shape[:-1], N)


def _w8_operands(x, wq, scale_, outlier_idx, w_out, bias) -> tuple:
    """The checked operands of an int8 Linear as the library takes them (no outlier columns: None), and M, N, K and the number of outlier columns."""
    require_device(x, "linear_w8")
    dtype = x.dtype
    if wq.dtype is not torch.int8 or scale_.dtype is not torch.float32:
        raise TypeError("linear_w8: wq must be int8 and scale float32")
    if dtype is not torch.bfloat16 and dtype is not torch.float16:
        raise TypeError(f"linear_w8: x must be bfloat16 or float16, got {x.dtype}")
    x2 = _as_2d(x)
    M, K = x2.shape
    if wq.dim() != 2 or wq.shape[1] != K:
        raise ValueError(f"linear_w8: x has {K} input features, wq is {tuple(wq.shape)}")
    N = wq.shape[0]
    if scale_.shape != (N,):
        raise ValueError(f"linear_w8: scale must have shape [{N}], got {tuple(scale_.shape)}")
    index = x.get_device()
    if (index < 0 or wq.get_device() != index or scale_.get_device() != index or outlier_idx is not None and outlier_idx.get_device() != index
            or w_out is not None and w_out.get_device() != index or bias is not None and bias.get_device() != index):
        for name, t in (("wq", wq), ("scale", scale_), ("outlier_idx", outlier_idx), ("w_out", w_out), ("bias", bias)):
            if t is not None and t.device != x.device:
                raise ValueError(f"linear_w8: x is on {x.device}, {name} on {t.device}")
    if bias is not None:
        if bias.shape != (N,) or bias.dtype is not dtype:
            raise ValueError("linear_w8: bias must have shape [N] and the dtype of x")
        bias = bias.contiguous()
    n_out = 0 if outlier_idx is None else outlier_idx.numel()
    if n_out == 0:
        return (x2, wq.contiguous(), scale_.contiguous(), None, None, bias), (M, N, K, 0)
    if outlier_idx.dtype is not torch.int32 or w_out is None or w_out.shape != (N, n_out) or w_out.dtype is not dtype:
        raise ValueError("linear_w8: outlier_idx must be int32 [n_out] and w_out [N, n_out] in the dtype of x")
    if n_out > K:
        raise ValueError(f"linear_w8: {n_out} outlier columns for K = {K}")
    return (x2, wq.contiguous(), scale_.contiguous(), outlier_idx.contiguous(), w_out.contiguous(), bias), (M, N, K, n_out)


def _w8_ranks(calls: Sequence[tuple]) -> tuple:
    ranks, keep = (W8Rank * len(calls))(), []
    for rank, call in zip(ranks, calls):
        ops, (M, N, K, n_out) = _w8_operands(*call[:6])
        x2 = ops[0]
        y = torch.empty((M, N), dtype=x2.dtype, device=x2.device)
        keep.append((ops, y))
        rank.x, rank.wq, rank.scale, rank.outlier_idx, rank.w_out, rank.bias = (None if t is None else t.data_ptr() for t in ops)
        rank.y = y.data_ptr()
    return ranks, keep, (n_out, M, N, K, _ld(x2), K, max(n_out, 1), N, dtype_code(x2.dtype))


def linear_w8_ranks(calls: Sequence[tuple]) -> list:
    """`linear_w8(x, wq, scale, outlier_idx, w_out, bias, act)` for the operands of several ranks."""
    x, act = calls[0][0], calls[0][6] if len(calls[0]) > 6 else ACT_NONE
    with _on_device(x.device):
        ranks, keep, dims = _w8_ranks(calls)
        _check(lib().tpamd_linear_w8_ranks(len(calls), ranks, *dims, act, ctypes.c_void_p(current_stream_ptr(x.device))), "tpamd_linear_w8_ranks")
    return [y.view(*x.shape[:-1], y.shape[1]) for _, y in keep]


def linear_w8_sum_ranks(calls: Sequence[tuple]) -> Optional[list]:
    """The sum of two ranks' `linear_w8`, for each a tensor of its own; None where no launch of both adds it up."""
    x = calls[0][0]
    with _on_device(x.device):
        ranks, keep, dims = _w8_ranks(calls)
        rc = lib().tpamd_linear_w8_sum_ranks(ranks, *dims, ctypes.c_void_p(current_stream_ptr(x.device)))
    if rc == -2:
        return None
    _check(rc, "tpamd_linear_w8_sum_ranks")
    return [y.view(*x.shape[:-1], y.shape[1]) for _, y in keep]
