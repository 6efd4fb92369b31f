"""ctypes binding of libgdn_hip.so (the C ABI declared in include/gdn_hip.h).

The library is loaded from the package's ``lib/`` directory; it is built
in-tree by ``myvllm_amd.build.build()``.  ``MYVLLM_AMD_LIB`` in the environment
names another build of the same library instead (the host-AddressSanitizer
build of ``myvllm_amd.build.build_asan()``, for the C-ABI tests).  There is no
fallback: if the library is missing every op raises.
"""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os
import threading

import torch

LIB_PATH = os.environ.get("MYVLLM_AMD_LIB") or os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib",
                                                            "libgdn_hip.so")
BINDING_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib", "_gdn_binding.so")
ABI_VERSION = 1
MAX_NDIM = 4

# flags of gdn_chunk_prefill_ex (include/gdn_hip.h)
PREFILL_ZERO_INIT = 1
PREFILL_ACCUM_STATE = 2
PREFILL_ACCUM_OUT = 4

DTYPE_CODES = {
    torch.float32: 0,
    torch.bfloat16: 1,
    torch.float16: 2,
    torch.int32: 3,
    torch.int64: 4,
}

EXPORTED_SYMBOLS = (
    "gdn_recurrent_step",
    "gdn_chunk_prefill",
    "gdn_chunk_prefill_ex",
    "gdn_chunk_prefill_workspace_size",
    "gdn_chunk_prefill_split",
    "gdn_chunk_prefill_split_ex",
    "causal_conv1d_varlen",
    "causal_conv1d_step",
    "gdn_decode_step_fused",
    "gdn_decode_step_fused_norm",
    "gdn_linear",
    "causal_conv1d_varlen_qknorm",
    "gdn_rms_norm_gated",
    "gdn_gating",
    "flash_attention_varlen",
    "flash_attention_varlen_any_dim",
    "paged_attention_prefill",
    "paged_attention_prefill_workspace_size",
    "paged_attention_prefill_split",
    "paged_attention_decode_workspace_size",
    "paged_attention_decode",
    "paged_attention_decode_noalloc",
    "gdn_hbm_copy",
    "gdn_strerror",
    "gdn_abi_version",
)


class GdnTensor(ctypes.Structure):
    """Mirror of ``struct gdn_tensor``."""

    _fields_ = [
        ("data", ctypes.c_void_p),
        ("dtype", ctypes.c_int32),
        ("ndim", ctypes.c_int32),
        ("shape", ctypes.c_int64 * MAX_NDIM),
        ("stride", ctypes.c_int64 * MAX_NDIM),
    ]


class GdnError(RuntimeError):
    """A non-zero return code of the C ABI (negative: validation, positive: HIP)."""

    def __init__(self, fn: str, code: int, msg: str):
        super().__init__(f"{fn} failed with code {code}: {msg}")
        self.code = code


_lib = None
_fast = None  # the native call path (csrc/binding.cpp), bound to the loaded library
_lock = threading.Lock()
_PT = ctypes.POINTER(GdnTensor)


def _load_binding(lib: ctypes.CDLL):
    if not os.path.exists(BINDING_PATH):
        raise RuntimeError(f"{BINDING_PATH} is missing: build the library first (see load())")
    loader = importlib.machinery.ExtensionFileLoader("_gdn_binding", BINDING_PATH)
    mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("_gdn_binding", loader))
    loader.exec_module(mod)
    mod.bind({n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in EXPORTED_SYMBOLS})
    return mod


def load() -> ctypes.CDLL:
    """Load (once) and type the shared library; raises if it has not been built."""
    global _lib, _fast
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it first with `python -c 'import __graft_entry__ as g; g.build()'` "
                "(or `python myvllm_amd/build.py`); there is no CPU fallback"
            )
        lib = ctypes.CDLL(LIB_PATH)
        lib.gdn_abi_version.restype = ctypes.c_int
        lib.gdn_abi_version.argtypes = []
        lib.gdn_strerror.restype = ctypes.c_char_p
        lib.gdn_strerror.argtypes = [ctypes.c_int]
        lib.gdn_recurrent_step.restype = ctypes.c_int
        lib.gdn_recurrent_step.argtypes = [_PT] * 8 + [ctypes.c_float, ctypes.c_void_p]
        lib.gdn_chunk_prefill.restype = ctypes.c_int
        lib.gdn_chunk_prefill.argtypes = [_PT] * 9 + [ctypes.c_float, ctypes.c_int32, ctypes.c_void_p]
        lib.gdn_chunk_prefill_ex.restype = ctypes.c_int
        lib.gdn_chunk_prefill_ex.argtypes = [_PT] * 9 + [ctypes.c_float] + [ctypes.c_int32] * 4 + [ctypes.c_void_p]
        lib.gdn_chunk_prefill_workspace_size.restype = ctypes.c_int64
        lib.gdn_chunk_prefill_workspace_size.argtypes = [ctypes.c_int64] * 6
        lib.gdn_chunk_prefill_split.restype = ctypes.c_int
        lib.gdn_chunk_prefill_split.argtypes = [_PT] * 10 + [ctypes.c_float, ctypes.c_int32, ctypes.c_void_p]
        lib.gdn_chunk_prefill_split_ex.restype = ctypes.c_int
        lib.gdn_chunk_prefill_split_ex.argtypes = [_PT] * 10 + [ctypes.c_float] + [ctypes.c_int32] * 2 + \
            [ctypes.c_void_p]
        lib.causal_conv1d_varlen.restype = ctypes.c_int
        lib.causal_conv1d_varlen.argtypes = [_PT] * 6 + [ctypes.c_void_p]
        lib.causal_conv1d_step.restype = ctypes.c_int
        lib.causal_conv1d_step.argtypes = [_PT] * 5 + [ctypes.c_void_p]
        lib.gdn_decode_step_fused.restype = ctypes.c_int
        lib.gdn_decode_step_fused.argtypes = [_PT] * 11 + [ctypes.c_int32, ctypes.c_float, ctypes.c_void_p]
        lib.gdn_decode_step_fused_norm.restype = ctypes.c_int
        lib.gdn_decode_step_fused_norm.argtypes = [_PT] * 13 + [ctypes.c_int32, ctypes.c_float, ctypes.c_float,
                                                                ctypes.c_void_p]
        lib.gdn_linear.restype = ctypes.c_int
        lib.gdn_linear.argtypes = [_PT] * 3 + [ctypes.c_void_p]
        lib.causal_conv1d_varlen_qknorm.restype = ctypes.c_int
        lib.causal_conv1d_varlen_qknorm.argtypes = [_PT] * 6 + [ctypes.c_int64, ctypes.c_void_p]
        lib.gdn_rms_norm_gated.restype = ctypes.c_int
        lib.gdn_rms_norm_gated.argtypes = [_PT] * 4 + [ctypes.c_float, ctypes.c_void_p]
        lib.gdn_gating.restype = ctypes.c_int
        lib.gdn_gating.argtypes = [_PT] * 6 + [ctypes.c_void_p]
        lib.flash_attention_varlen.restype = ctypes.c_int
        lib.flash_attention_varlen.argtypes = [_PT] * 5 + [ctypes.c_int64, ctypes.c_float, ctypes.c_int32,
                                                           ctypes.c_void_p]
        lib.flash_attention_varlen_any_dim.restype = ctypes.c_int
        lib.flash_attention_varlen_any_dim.argtypes = lib.flash_attention_varlen.argtypes
        lib.paged_attention_prefill.restype = ctypes.c_int
        lib.paged_attention_prefill.argtypes = [_PT] * 7 + [ctypes.c_int64, ctypes.c_float, ctypes.c_void_p]
        lib.paged_attention_prefill_workspace_size.restype = ctypes.c_int64
        lib.paged_attention_prefill_workspace_size.argtypes = [ctypes.c_int64] * 6
        lib.paged_attention_prefill_split.restype = ctypes.c_int
        lib.paged_attention_prefill_split.argtypes = [_PT] * 8 + [ctypes.c_int64, ctypes.c_float, ctypes.c_void_p]
        lib.paged_attention_decode_workspace_size.restype = ctypes.c_int64
        lib.paged_attention_decode_workspace_size.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64,
                                                              ctypes.c_int32]
        lib.paged_attention_decode.restype = ctypes.c_int
        lib.paged_attention_decode.argtypes = [_PT] * 7 + [ctypes.c_int32, ctypes.c_float, ctypes.c_void_p]
        lib.paged_attention_decode_noalloc.restype = ctypes.c_int
        lib.gdn_hbm_copy.restype = ctypes.c_int
        lib.gdn_hbm_copy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64, ctypes.c_int32,
                                     ctypes.c_void_p]
        lib.paged_attention_decode_noalloc.argtypes = [_PT] * 6 + [ctypes.c_int32, ctypes.c_float, ctypes.c_void_p]
        if lib.gdn_abi_version() != ABI_VERSION:
            raise RuntimeError(f"{LIB_PATH} has ABI {lib.gdn_abi_version()}, expected {ABI_VERSION}; rebuild it")
        _fast = _load_binding(lib)
        _lib = lib
        return lib


def _load_fast():
    load()
    return _fast


def workspace_size(fn: str, *sizes: int) -> int:
    """One of the library's ``*_workspace_size`` functions."""
    return getattr(_fast or _load_fast(), fn)(*sizes)


def strerror(code: int) -> str:
    return load().gdn_strerror(int(code)).decode()


def describe(t: torch.Tensor | None) -> GdnTensor:
    """Descriptor of a tensor (device pointer, dtype code, shape, element strides)."""
    d = GdnTensor()
    if t is None:
        return d
    if t.dim() > MAX_NDIM:
        raise ValueError(f"tensors of rank > {MAX_NDIM} are not supported")
    d.data = t.data_ptr() if t.numel() > 0 else None
    d.dtype = DTYPE_CODES.get(t.dtype, -1)
    d.ndim = t.dim()
    for i in range(t.dim()):
        d.shape[i] = t.shape[i]
        d.stride[i] = t.stride(i)
    return d


def call(fn: str, *args) -> None:
    """Entry point `fn` on tensors (None: a null descriptor) and scalars, on the
    current stream of the first tensor's device; raises on a non-zero code.
    Plain tensors go through the native call path, others through ctypes."""
    lib = _lib or load()
    code = getattr(_fast, fn)(*args)
    if code is None:
        code = getattr(lib, fn)(*(describe(a) if isinstance(a, torch.Tensor) else a for a in args),
                                stream_handle(args[0].device))
    if code:
        raise GdnError(fn, code, strerror(code))


def check(fn: str, code: int) -> None:
    if code != 0:
        raise GdnError(fn, code, strerror(code))


def vec16_ok(t: torch.Tensor) -> bool:
    """Whether the kernels can read t with 16-byte vector accesses: unit inner
    stride, 16-byte aligned data and outer strides."""
    ok = (_fast or _load_fast()).vec16_ok(t)
    if ok is not None:
        return ok
    es = t.element_size()
    return t.stride(-1) == 1 and t.data_ptr() % 16 == 0 and all((t.stride(i) * es) % 16 == 0 for i in range(t.dim() - 1))


def vec16(t: torch.Tensor) -> torch.Tensor:
    """t itself when the kernels can read it with 16-byte vector accesses, else a
    contiguous copy (also of a contiguous one at a misaligned address): the
    reference passes every stride to its kernels, so any strided input is
    accepted, at the cost of a copy when it is misaligned."""
    return t if vec16_ok(t) else t.clone(memory_format=torch.contiguous_format)


def same_device(*tensors: torch.Tensor) -> bool:
    """Whether all of them are plain tensors on one HIP device."""
    return (_fast or _load_fast()).same_device(*tensors) >= 0


def require_device(*tensors: torch.Tensor) -> torch.device:
    """All tensors must live on one HIP device (the kernels dereference the pointers)."""
    if same_device(*tensors):
        return next(t for t in tensors if t is not None).device
    dev = None
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise ValueError("myvllm_amd ops take GPU tensors only (got a tensor on %s)" % t.device)
        if dev is None:
            dev = t.device
        elif t.device != dev:
            raise ValueError(f"tensors on different devices: {dev} and {t.device}")
    return dev


def stream_handle(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream
