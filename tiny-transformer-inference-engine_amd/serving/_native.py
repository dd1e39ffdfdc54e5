"""ctypes binding of libpagedkv.so (the HIP kernels behind the C ABI in
include/pagedkv.h).

The library is required: every function here raises RuntimeError when it is
missing or when a tensor is not on a ROCm device. There is no CPU fallback.
"""
from __future__ import annotations

import contextlib
import ctypes
import importlib.machinery
import importlib.util
import os
import threading

import torch

_PKG_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB_PATH = os.path.join(_PKG_ROOT, "lib", "libpagedkv.so")
BIND_PATH = os.path.join(_PKG_ROOT, "lib", "_pkvbind.so")

DTYPE_CODES = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
# OR-ed into a dtype code: the K/V pools hold fp8 e4m3 (torch.float8_e4m3fn)
# while Q, out and appended rows keep the coded type
PKV_KV_FP8 = 0x100
FP8_KV_DTYPE = torch.float8_e4m3fn

PKV_ERR_INVALID = -1
PKV_ERR_UNSUPPORTED = -2
PKV_ERR_WORKSPACE = -3
PKV_ERR_HIP = -4

PKV_STATUS_BAD_SLOT = 1
PKV_STATUS_BAD_BLOCK = 2
PKV_STATUS_SHORT_TABLE = 4
PKV_STATUS_BAD_QLOC = 8
PKV_STATUS_BAD_POS = 16
PKV_STATUS_NONFINITE = 32
PKV_STATUS_BAD_DISTRIBUTION = 64
PKV_STATUS_SAMPLE_OVERFLOW = 128
PKV_STATUS_DIRTY_WORKSPACE = 256
PKV_STATUS_STALLED = 512
# part_tokens values selecting a persistent decode kernel (every workgroup an
# equal share of all sequences' chunks): PART_PERSISTENT and PART_STATIC the
# register-staged kernel (also the automatic choice for long context
# bounds), PART_STREAM the wavefront-specialised one (producer wavefronts
# streaming K/V into LDS by LDS-DMA, consumer wavefronts computing) where it
# applies, else the register-staged one
PART_PERSISTENT = -1
PART_STATIC = -2
PART_STREAM = -3

# epilogue values of pkv_linear_tiles
EPILOGUE_NONE = 0
EPILOGUE_SWIGLU = 1
EPILOGUE_RESIDUAL = 2

_lib = None
_calls = None
_lock = threading.Lock()

_c_i64 = ctypes.c_int64
_c_int = ctypes.c_int
_c_vp = ctypes.c_void_p
_c_size = ctypes.c_size_t
_c_float = ctypes.c_float

_SIGNATURES = {
    "pkv_version": ([], _c_int),
    "pkv_last_error": ([], ctypes.c_char_p),
    "pkv_append": ([_c_vp, _c_vp, _c_i64, _c_vp, _c_vp, _c_vp, _c_i64, _c_i64,
                    _c_int, _c_vp, _c_vp], _c_int),
    "pkv_append_from_table": ([_c_vp, _c_vp, _c_i64, _c_int, _c_vp, _c_vp,
                               _c_vp, _c_int, _c_vp, _c_vp, _c_int, _c_i64,
                               _c_i64, _c_int, _c_vp, _c_vp], _c_int),
    "pkv_gather": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_int, _c_vp, _c_int,
                    _c_int, _c_i64, _c_int, _c_vp, _c_vp], _c_int),
    "pkv_attention_workspace_bytes": ([_c_int, _c_int, _c_int, _c_int, _c_int,
                                       _c_int, _c_int, _c_int, _c_int, _c_int],
                                      _c_size),
    "pkv_paged_attention": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_int,
                             _c_vp, _c_int, _c_vp, _c_vp, _c_int, _c_int, _c_int,
                             _c_int, _c_int, _c_int, _c_int, _c_float, _c_int,
                             _c_int, _c_int, _c_vp, _c_size, _c_vp, _c_vp],
                            _c_int),
    "pkv_paged_attention_append": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_int,
                                    _c_vp, _c_int, _c_vp, _c_vp, _c_int, _c_int, _c_int,
                                    _c_int, _c_int, _c_int, _c_int, _c_float, _c_int,
                                    _c_int, _c_int, _c_vp, _c_vp, _c_vp, _c_vp, _c_size,
                                    _c_vp, _c_vp], _c_int),
    "pkv_paged_attention_noalloc": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_int,
                                     _c_vp, _c_int, _c_vp, _c_vp, _c_int, _c_int, _c_int,
                                     _c_int, _c_int, _c_int, _c_int, _c_float, _c_int,
                                     _c_int, _c_int, _c_vp, _c_vp], _c_int),
    "pkv_rms_norm": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_int, _c_i64, _c_i64,
                      _c_float, _c_int, _c_vp], _c_int),
    "pkv_rope": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_i64, _c_i64, _c_vp,
                  _c_vp, _c_vp, _c_int, _c_i64, _c_int, _c_int, _c_int, _c_int, _c_vp, _c_vp],
                 _c_int),
    "pkv_silu_mul": ([_c_vp, _c_vp, _c_vp, _c_i64, _c_i64, _c_i64, _c_i64, _c_int, _c_vp],
                     _c_int),
    "pkv_linear": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_i64, _c_i64, _c_i64, _c_int,
                    _c_vp], _c_int),
    "pkv_linear_swiglu": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_i64, _c_i64, _c_i64, _c_int,
                           _c_vp], _c_int),
    "pkv_linear_rope_qkv": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_i64, _c_i64,
                             _c_vp, _c_vp, _c_vp, _c_int, _c_int, _c_int, _c_int, _c_int,
                             _c_vp, _c_vp], _c_int),
    "pkv_linear_residual": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_i64, _c_i64, _c_i64, _c_int,
                             _c_vp], _c_int),
    "pkv_linear_swiglu_rmsnorm": ([_c_vp, _c_vp, _c_vp, _c_float, _c_vp, _c_vp, _c_i64, _c_i64,
                                   _c_i64, _c_i64, _c_int, _c_vp], _c_int),
    "pkv_linear_rope_qkv_rmsnorm": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_float, _c_vp, _c_vp,
                                     _c_i64, _c_i64, _c_i64, _c_vp, _c_vp, _c_vp, _c_int, _c_int,
                                     _c_int, _c_int, _c_int, _c_vp, _c_vp], _c_int),
    "pkv_linear_tiles": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_i64, _c_i64, _c_i64, _c_int,
                          _c_int, _c_vp], _c_int),
    "pkv_linear_tiles_rope_qkv": ([_c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_vp, _c_i64, _c_i64,
                                   _c_i64, _c_vp, _c_vp, _c_vp, _c_int, _c_int, _c_int, _c_int,
                                   _c_int, _c_vp, _c_vp], _c_int),
    "pkv_argmax_workspace_bytes": ([_c_i64, _c_i64, _c_int], _c_size),
    "pkv_argmax_rows": ([_c_vp, _c_vp, _c_i64, _c_i64, _c_i64, _c_int, _c_vp, _c_size, _c_vp],
                        _c_int),
    "pkv_sample_rows": ([_c_vp, _c_vp, _c_i64, _c_i64, _c_i64, _c_float, _c_int, _c_float,
                         _c_vp, _c_int, _c_vp, _c_vp], _c_int),
    "pkv_stream_read": ([_c_vp, _c_i64, _c_vp, _c_int, _c_vp], _c_int),
}

EXPORTED = tuple(_SIGNATURES)


def lib():
    """Load (once) and return the ctypes handle of libpagedkv.so."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not os.path.exists(LIB_PATH):
                raise RuntimeError(
                    f"libpagedkv.so not found at {LIB_PATH}; build it with "
                    "`python tiny-transformer-inference-engine_amd/build_native.py` "
                    "(or __graft_entry__.build())")
            handle = ctypes.CDLL(LIB_PATH)
            for name, (args, res) in _SIGNATURES.items():
                fn = getattr(handle, name)
                fn.argtypes = args
                fn.restype = res
            _lib = handle
    return _lib


def calls():
    """The library's entry points as the wrappers call them: the module
    _pkvbind (csrc/bind.cpp), bound to lib()'s instance, or lib() itself (the
    same calls through ctypes, some 4 us slower each) where that module was not
    built or this interpreter does not load it."""
    global _calls
    if _calls is not None:
        return _calls
    handle = lib()
    with _lock:
        if _calls is None:
            loader = importlib.machinery.ExtensionFileLoader("_pkvbind", BIND_PATH)
            spec = importlib.util.spec_from_file_location("_pkvbind", BIND_PATH, loader=loader)
            try:
                mod = importlib.util.module_from_spec(spec)
                loader.exec_module(mod)
            except ImportError:  # no such file, or another interpreter's
                mod = handle
            else:
                mod.bind({name: ctypes.cast(getattr(handle, name), ctypes.c_void_p).value
                          for name in _SIGNATURES})
            _calls = mod
    return _calls


def is_available() -> bool:
    """True when the library loads and a ROCm device is visible."""
    try:
        calls()
    except (RuntimeError, OSError):
        return False
    return torch.cuda.is_available()


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = lib().pkv_last_error().decode(errors="replace")
        if rc == -1:
            raise ValueError(f"{what}: {msg}")
        if rc == -2:
            raise NotImplementedError(f"{what}: {msg}")
        raise RuntimeError(f"{what} failed ({rc}): {msg}")


def require_device(*tensors: torch.Tensor, what: str = "paged kv op") -> None:
    for t in tensors:
        if not t.is_cuda:
            raise RuntimeError(
                f"{what} requires tensors on a ROCm GPU device (got {t.device}); "
                "the HIP library has no CPU path")


def dtype_code(dtype: torch.dtype) -> int:
    try:
        return DTYPE_CODES[dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {dtype}; expected float32, float16 or bfloat16")


def kv_code(q_dtype: torch.dtype, pool_dtype: torch.dtype) -> int:
    """dtype argument of a call with Q (or appended rows) of q_dtype and pools
    of pool_dtype: pools share the 16/32-bit type, or are fp8 e4m3."""
    if pool_dtype == FP8_KV_DTYPE:
        return dtype_code(q_dtype) | PKV_KV_FP8
    if pool_dtype != q_dtype:
        raise TypeError(f"pool dtype {pool_dtype} with rows of {q_dtype}: pools share the "
                        "rows' dtype or are float8_e4m3fn")
    return dtype_code(q_dtype)


# the current stream's handle by device index, without building a Stream object
# (2.0 us against 0.1 a call)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_ptr(device: torch.device) -> int:
    if _raw_stream is None or device.index is None:
        return torch.cuda.current_stream(device).cuda_stream
    return _raw_stream(device.index)


def ptr(t) -> int | None:
    return None if t is None else t.data_ptr()


class Workspace:
    """Per-device scratch for split-K partials and the persistent kernel's
    per-sequence records (slot "attention") and for the split-row argmax
    kernel's counters and key words (slot "argmax"), one buffer per
    (device, slot), grown on demand and reused (the library never
    allocates). Allocation goes through torch's caching allocator, so it is
    stream-ordered on the current stream; calls on other streams need their
    own Workspace."""

    def __init__(self):
        self._bufs: dict[tuple[int, str], torch.Tensor] = {}

    def get(self, device: torch.device, nbytes: int,
            slot: str = "attention") -> torch.Tensor | None:
        if nbytes == 0:
            return None
        idx = device.index if device.index is not None else torch.cuda.current_device()
        buf = self._bufs.get((idx, slot))
        if buf is None or buf.numel() < nbytes:
            # grow geometrically so ragged batches do not reallocate every step
            size = max(nbytes, 0 if buf is None else 2 * buf.numel())
            # zero-filled once: the kernels' arrival counters (and the argmax
            # key words) must start at zero, and every call leaves them zero;
            # partials and records are written before they are read
            buf = torch.zeros(size, dtype=torch.uint8, device=device)
            self._bufs[(idx, slot)] = buf
        return buf


WORKSPACE = Workspace()

_scopes = threading.local()


def current_workspace() -> Workspace:
    """The Workspace the attention wrappers use on this thread: the innermost
    workspace_scope, else the process-wide WORKSPACE."""
    stack = getattr(_scopes, "stack", None)
    return stack[-1] if stack else WORKSPACE


@contextlib.contextmanager
def workspace_scope(ws: Workspace):
    """Route the attention wrappers' scratch to `ws` inside the block. A HIP
    graph captures the raw address of the buffer it is given, so a captured
    step needs a workspace no later eager call can grow (and thereby free);
    serving.graph_step holds one per graph for the graph's lifetime."""
    stack = getattr(_scopes, "stack", None)
    if stack is None:
        stack = _scopes.stack = []
    stack.append(ws)
    try:
        yield ws
    finally:
        stack.pop()
