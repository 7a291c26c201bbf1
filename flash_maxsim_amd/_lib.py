"""ctypes binding of libflashmaxsim.so (declarations in include/fmx.h).

torch is imported first so the HIP runtime bundled with torch is already
loaded: libflashmaxsim's libamdhip64.so.7 dependency then resolves to that same
runtime, and torch's streams and device pointers are valid inside the library.
"""

from __future__ import annotations

import ctypes
from pathlib import Path

import torch  # noqa: F401  (must load the HIP runtime before the library)

LIB_PATH = Path(__file__).resolve().with_name("libflashmaxsim.so")

FMX_DTYPE_F16 = 0
FMX_DTYPE_BF16 = 1
FMX_DTYPE_F32 = 2

_i64 = ctypes.c_int64
_ptr = ctypes.c_void_p
_int = ctypes.c_int
_size = ctypes.c_size_t

# name -> (restype, argtypes)
_SIGNATURES = {
    "fmx_version": (ctypes.c_char_p, []),
    "fmx_last_error": (ctypes.c_char_p, []),
    "fmx_fwd": (
        _int,
        [_int, _ptr, _i64, _i64, _ptr, _i64, _i64, _ptr, _ptr, _i64, _i64, _ptr,
         _i64, _i64, _i64, _i64, _i64, _int, _ptr, _size, _ptr],
    ),
    "fmx_fwd_workspace_bytes": (_size, [_i64, _i64, _i64, _i64, _i64]),
    "fmx_fwd_reads_f32": (_int, [_i64, _i64]),
    "fmx_fwd_noalloc": (
        _int,
        [_int, _ptr, _i64, _i64, _ptr, _i64, _i64, _ptr, _ptr, _i64, _i64, _ptr,
         _i64, _i64, _i64, _i64, _i64, _int, _ptr],
    ),
    "fmx_fwd_int8": (
        _int,
        [_ptr, _i64, _ptr, _i64, _i64, _ptr, _ptr, _i64, _ptr, _ptr,
         _i64, _i64, _i64, _i64, _ptr, _size, _ptr],
    ),
    "fmx_fwd_int8_workspace_bytes": (_size, [_i64, _i64, _i64, _i64]),
    "fmx_fwd_sparse": (
        _int,
        [_int, _ptr, _i64, _i64, _ptr, _i64, _i64, _ptr, _i64, _i64, _i64, _ptr, _ptr,
         _i64, _i64, _i64, _ptr, _size, _ptr],
    ),
    "fmx_fwd_sparse_workspace_bytes": (_size, [_i64, _i64, _i64, _i64]),
    "fmx_quantize_int8": (
        _int,
        [_int, _ptr, _i64, _i64, _i64, _i64, _i64, _ptr, _ptr, _i64, _ptr, _i64, _ptr, _ptr, _i64, _ptr],
    ),
    "fmx_dequantize_int8": (_int, [_ptr, _ptr, _ptr, _i64, _i64, _ptr, _ptr]),
    "fmx_packed_layout": (_int, [_ptr, _i64, _i64, _ptr, _ptr, _ptr, _ptr]),
    "fmx_pack_rows": (_int, [_ptr, _i64, _i64, _i64, _i64, _i64, _ptr, _ptr, _i64, _ptr, _ptr]),
    "fmx_fwd_packed": (
        _int,
        [_int, _ptr, _i64, _i64, _ptr, _i64, _i64, _ptr, _ptr, _ptr, _ptr, _i64, _i64, _i64, _ptr, _size, _ptr],
    ),
    "fmx_fwd_packed_workspace_bytes": (_size, [_i64, _i64, _i64, _i64]),
    "fmx_fwd_int8_packed": (
        _int,
        [_ptr, _i64, _i64, _ptr, _i64, _ptr, _ptr, _i64, _ptr, _ptr, _ptr, _ptr, _i64, _i64, _i64, _ptr, _size, _ptr],
    ),
    "fmx_fwd_int8_packed_workspace_bytes": (_size, [_i64, _i64, _i64, _i64]),
    "fmx_topk": (_int, [_ptr, _i64, _i64, _i64, _i64, _ptr, _ptr, _i64, _ptr, _size, _ptr]),
    "fmx_topk_workspace_bytes": (_size, [_i64, _i64, _i64]),
    "fmx_fwd_topk": (
        _int,
        [_int, _ptr, _i64, _ptr, _i64, _i64, _ptr, _i64, _i64, _i64, _i64, _i64, _ptr, _ptr, _ptr, _ptr, _size,
         _ptr],
    ),
    "fmx_fwd_topk_workspace_bytes": (_size, [_i64, _i64, _i64, _i64, _i64]),
    "fmx_bwd": (
        _int,
        [_int, _ptr, _i64, _ptr, _i64, _i64, _ptr, _ptr, _ptr, _ptr,
         _i64, _i64, _i64, _i64, _ptr, _size, _ptr],
    ),
    "fmx_bwd_workspace_bytes": (_size, [_i64, _i64, _i64, _i64]),
    "fmx_bwd_batched": (
        _int,
        [_int, _ptr, _i64, _i64, _ptr, _i64, _i64, _ptr, _ptr, _ptr, _i64, _i64, _ptr, _ptr,
         _i64, _i64, _i64, _i64, _i64, _ptr, _size, _ptr],
    ),
    "fmx_bwd_batched_f32": (
        _int,
        [_ptr, _i64, _i64, _ptr, _i64, _i64, _ptr, _ptr, _ptr, _i64, _i64, _ptr, _ptr,
         _i64, _i64, _i64, _i64, _i64, _ptr, _size, _ptr],
    ),
    "fmx_convert_rows": (_int, [_int, _ptr, _i64, _i64, _i64, _i64, _i64, _ptr, _int, _ptr, _i64, _ptr]),
    "fmx_bwd_batched_workspace_bytes": (_size, [_i64, _i64, _i64, _i64, _i64]),
}

EXPORTED = tuple(_SIGNATURES)

_lib: ctypes.CDLL | None = None


def load() -> ctypes.CDLL:
    """Loads libflashmaxsim.so once; raises if it was never built."""
    global _lib
    if _lib is None:
        if not LIB_PATH.exists():
            raise RuntimeError(
                f"{LIB_PATH} is missing: build the HIP extension first "
                "(`python -m flash_maxsim_amd.build`, needs hipcc for gfx950)"
            )
        lib = ctypes.CDLL(str(LIB_PATH))
        for name, (res, args) in _SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        _lib = lib
    return _lib


_native = None


def native():
    """The native host path (csrc/native.cpp): one function per ordinary call,
    each returning None where the call has to take the Python path."""
    global _native
    if _native is None:
        load()  # names what is missing; the module links to the same library
        from . import _native as module

        _native = module
    return _native


def check(rc: int) -> None:
    if rc != 0:
        msg = load().fmx_last_error().decode(errors="replace")
        raise RuntimeError(f"flash_maxsim_amd: {msg} (code {rc})")


def ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def stream_of(t: torch.Tensor) -> int:
    return torch.cuda.current_stream(t.device).cuda_stream


def dtype_code(t: torch.Tensor) -> int:
    if t.dtype == torch.float16:
        return FMX_DTYPE_F16
    if t.dtype == torch.bfloat16:
        return FMX_DTYPE_BF16
    raise TypeError(f"kernel operands must be float16 or bfloat16, got {t.dtype}")


def plain(*tensors: torch.Tensor) -> bool:
    """True when a kernel may take the place of torch ops on these tensors:
    ordinary strided GPU tensors of one device, with nothing watching the ops
    (autograd in either mode, tracing, compilation, function transforms,
    dispatch or function modes)."""
    dev = tensors[0].device
    for t in tensors:
        if (type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter) or not t.is_cuda or t.device != dev:
            return False
        if t.layout is not torch.strided or t.is_neg() or (t.requires_grad and torch.is_grad_enabled()):
            return False
    return not (
        torch.compiler.is_compiling()
        or torch._C._get_tracing_state() is not None
        or torch._C._functorch.maybe_current_level() is not None
        or torch.autograd.forward_ad._current_level >= 0
        or torch._C._len_torch_dispatch_stack()
        or torch._C._len_torch_function_stack()
    )


def workspace(nbytes: int, device: torch.device) -> torch.Tensor | None:
    if nbytes == 0:
        return None
    return torch.empty((nbytes + 3) // 4, dtype=torch.float32, device=device)
