"""ctypes binding of libtileops_hip.so, the C-ABI library of gfx950 kernels.

The declarations mirror include/tileops_hip.h.  Kernel classes call the
``tileops_*`` functions with raw device pointers (``Tensor.data_ptr()``) and
the current HIP stream of the tensors' device, so launches are asynchronous
and ordered with the surrounding PyTorch work.

There is no fallback: if the library is missing, or a tensor is not on a HIP
device, the call raises.
"""

from __future__ import annotations

import ctypes
import functools
import os
import threading
from pathlib import Path

import torch

__all__ = [
    "DTYPE_CODES",
    "LIB_PATH",
    "check",
    "dtype_code",
    "eager",
    "lib",
    "require_device",
    "stream_of",
]

LIB_PATH = Path(
    os.environ.get(
        "TILEOPS_HIP_LIB", str(Path(__file__).resolve().parent / "_native" / "libtileops_hip.so")
    )
)

# enum tileops_reduce_op (include/tileops_hip.h)
LOGSUMEXP, ARGMAX, ARGMIN = 0, 1, 2

DTYPE_CODES = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}

_c_i64 = ctypes.c_int64
_c_int = ctypes.c_int
_c_float = ctypes.c_float
_c_p = ctypes.c_void_p

# name -> (restype, argtypes); kept in the order of include/tileops_hip.h
SIGNATURES = {
    "tileops_version": (_c_int, []),
    "tileops_error_string": (ctypes.c_char_p, [_c_int]),
    "tileops_unary_fwd": (
        _c_int,
        [_c_int, _c_p, _c_p, _c_i64, _c_int, _c_float, _c_float, _c_int, _c_p],
    ),
    "tileops_isfp_fwd": (_c_int, [_c_int, _c_p, _c_p, _c_i64, _c_int, _c_p]),
    "tileops_gated_gelu_fwd": (_c_int, [_c_int, _c_p, _c_p, _c_i64, _c_i64, _c_int, _c_p]),
    "tileops_fused_add_layernorm_fwd": (
        _c_int,
        [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_i64, _c_i64, _c_float, _c_int, _c_int, _c_p],
    ),
    "tileops_logsumexp_fwd": (_c_int, [_c_p, _c_p, _c_i64, _c_i64, _c_int, _c_p]),
    "tileops_argreduce_fwd": (_c_int, [_c_p, _c_p, _c_i64, _c_i64, _c_int, _c_int, _c_p]),
    "tileops_reduce_workspace_bytes": (ctypes.c_size_t, [_c_i64, _c_i64, _c_int]),
    "tileops_reduce_fwd": (
        _c_int,
        [_c_int, _c_p, _c_p, _c_i64, _c_i64, _c_int, _c_p, ctypes.c_size_t, _c_p],
    ),
    "tileops_reduce_axis_workspace_bytes": (
        ctypes.c_size_t,
        [_c_int, _c_i64, _c_i64, _c_i64, _c_int, _c_int],
    ),
    "tileops_reduce_axis_fwd": (
        _c_int,
        [_c_int, _c_p, _c_p, _c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_p, ctypes.c_size_t, _c_p],
    ),
    "tileops_mha_fwd": (
        _c_int,
        [
            _c_p, _c_p, _c_p, _c_p, _c_p,
            _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64,
            _c_int, _c_float, _c_float, _c_int, _c_p,
        ],
    ),
    "tileops_mha_workspace_bytes": (
        ctypes.c_size_t,
        [_c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_int, _c_float],
    ),
    "tileops_mha_fwd_ws": (
        _c_int,
        [
            _c_p, _c_p, _c_p, _c_p, _c_p,
            _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64,
            _c_int, _c_float, _c_float, _c_int, _c_p, ctypes.c_size_t, _c_p,
        ],
    ),
    "tileops_mha_workspace_bytes_ex": (
        ctypes.c_size_t,
        [_c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_int, _c_float, _c_i64],
    ),
    "tileops_mha_fwd_ex": (
        _c_int,
        [
            _c_p, _c_p, _c_p, _c_p, _c_p,
            _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64,
            _c_int, _c_float, _c_float, _c_int, _c_i64, _c_p, ctypes.c_size_t, _c_p,
        ],
    ),
    "tileops_gdn_prefill_fwd": (
        _c_int,
        [
            _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p,
            _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64,
            _c_float, _c_int, _c_p, ctypes.c_size_t, _c_p,
        ],
    ),
    "tileops_gdn_prefill_workspace_bytes": (
        ctypes.c_size_t,
        [_c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64],
    ),
    "tileops_gdn_prefill_fwd_ex": (
        _c_int,
        [
            _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p,
            _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64,
            _c_float, _c_int, _c_i64, _c_p, ctypes.c_size_t, _c_p,
        ],
    ),
    "tileops_gdn_prefill_workspace_bytes_ex": (
        ctypes.c_size_t,
        [_c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64],
    ),
    "tileops_gdn_prefill_fwd_noalloc": (
        _c_int,
        [
            _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p,
            _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64,
            _c_float, _c_int, _c_p,
        ],
    ),
    "tileops_bitwise_not_fwd": (_c_int, [_c_p, _c_p, _c_i64, _c_int, _c_p]),
    "tileops_add_fwd": (_c_int, [_c_p, _c_p, _c_p, _c_int, _c_p, _c_p, _c_p, _c_float, _c_int, _c_p]),
    "tileops_lerp_fwd": (
        _c_int,
        [_c_p, _c_p, _c_p, _c_p, _c_int, _c_p, _c_p, _c_p, _c_p, _c_float, _c_int, _c_p],
    ),
    "tileops_gla_decode_fwd": (
        _c_int,
        [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_i64, _c_i64, _c_i64, _c_i64, _c_float,
         _c_int, _c_p],
    ),
    "tileops_gdn_decode_fwd": (
        _c_int,
        [_c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_p, _c_i64, _c_i64, _c_i64, _c_i64,
         _c_float, _c_int, _c_p],
    ),
}

_lib = None
_lock = threading.Lock()


def lib() -> ctypes.CDLL:
    """Load libtileops_hip.so once; raise if it has not been built."""
    global _lib
    if _lib is None:
        with _lock:
            if _lib is None:
                if not LIB_PATH.is_file():
                    raise RuntimeError(
                        f"tileops: HIP library not found at {LIB_PATH}; build it with "
                        "`make -C tile-ascendnpu-ops_amd/csrc` (or __graft_entry__.build())"
                    )
                handle = ctypes.CDLL(str(LIB_PATH))
                for name, (restype, argtypes) in SIGNATURES.items():
                    fn = getattr(handle, name)
                    fn.restype = restype
                    fn.argtypes = argtypes
                _lib = handle
    return _lib


def check(code: int, what: str) -> None:
    """Raise RuntimeError for a nonzero tileops return code."""
    if code != 0:
        msg = lib().tileops_error_string(code)
        raise RuntimeError(f"{what} failed ({code}): {msg.decode() if msg else 'unknown'}")


def dtype_code(dtype: torch.dtype) -> int:
    try:
        return DTYPE_CODES[dtype]
    except KeyError:
        raise ValueError(f"tileops HIP kernels do not support dtype {dtype}") from None


_HIP = torch.version.hip is not None


def require_device(*tensors: torch.Tensor) -> None:
    """Every tensor must live in HIP device memory (there is no host path)."""
    for t in tensors:
        if t is not None and not (_HIP and t.is_cuda):
            raise RuntimeError(
                f"tileops HIP kernels need tensors on a ROCm GPU, got device {t.device}"
            )


def stream_of(t: torch.Tensor) -> int:
    """Raw hipStream_t of the current PyTorch stream on ``t``'s device."""
    return torch._C._cuda_getCurrentRawStream(t.get_device())


_PLAIN = (torch.Tensor, torch.nn.Parameter)

# looked up once: a call of `eager` is 0.65 us of a 10 us host path
_is_compiling = torch.compiler.is_compiling
_tracing_state = torch._C._get_tracing_state
_dispatch_modes = torch._C._len_torch_dispatch_stack
_function_modes = torch._C._len_torch_function_stack
_functorch_level = torch._C._functorch.peek_interpreter_stack
_forward_ad = torch.autograd.forward_ad


def eager(*tensors: torch.Tensor) -> bool:
    """True when a call on ``tensors`` may run its launch function directly
    rather than through the ``torch.library`` custom op around it.

    The custom op exists for everything that must see one opaque operator:
    compilation and tracing, dispatch and function modes (fake tensors among
    them), tensor subclasses, functorch transforms, forward-mode and
    reverse-mode autograd, and lazy negations and zeros, whose storage does not
    hold the values until the dispatcher resolves them.  A plain eager call is
    none of these and gets the same result from the launch function; the
    dispatcher's Python round trip costs it about 7 us (Argmax [4, 128]: 17.0 ->
    9.8 us per call).
    """
    if (
        _is_compiling()
        or _tracing_state() is not None
        or _dispatch_modes()
        or _function_modes()
        or _functorch_level() is not None
        or _forward_ad._current_level >= 0
    ):
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if type(t) not in _PLAIN or (grad and t.requires_grad) or t.is_neg() or t._is_zerotensor():
            return False
    return True


@functools.lru_cache(maxsize=1024)
def _reduce_scratch(M: int, N: int, code: int) -> int:
    return lib().tileops_reduce_workspace_bytes(M, N, code)


def reduce_rows(op: int, x: torch.Tensor, y: torch.Tensor, M: int, N: int) -> int:
    """``tileops_reduce_fwd`` of ``x[M, N]`` into ``y[M]``, with the scratch its
    launch plan asks for taken from torch's allocator (none for most shapes)."""
    code = dtype_code(x.dtype)
    need = _reduce_scratch(M, N, code)
    ws = torch.empty(need, dtype=torch.uint8, device=x.device) if need else None
    return lib().tileops_reduce_fwd(
        op, x.data_ptr(), y.data_ptr(), M, N, code, ws.data_ptr() if need else None, need,
        stream_of(x))


@functools.lru_cache(maxsize=1024)
def _reduce_axis_scratch(op: int, outer: int, n: int, inner: int, ends: int, code: int) -> int:
    return lib().tileops_reduce_axis_workspace_bytes(op, outer, n, inner, ends, code)


def reduce_axis(op: int, x: torch.Tensor, y: torch.Tensor, outer: int, n: int, inner: int,
                ends: bool) -> int:
    """``tileops_reduce_axis_fwd`` of contiguous ``x[outer, n, inner]`` over n
    (into ``y[outer, inner]``) or over outer and inner (into ``y[n]``)."""
    code, ends = dtype_code(x.dtype), int(ends)
    need = _reduce_axis_scratch(op, outer, n, inner, ends, code)
    ws = torch.empty(need, dtype=torch.uint8, device=x.device) if need else None
    return lib().tileops_reduce_axis_fwd(
        op, x.data_ptr(), y.data_ptr(), outer, n, inner, ends, code,
        ws.data_ptr() if need else None, need, stream_of(x))
