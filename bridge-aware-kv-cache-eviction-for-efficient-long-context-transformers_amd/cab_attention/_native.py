"""ctypes binding of libcab_hip.so (the C ABI declared in include/cab_hip.h).

There is exactly one implementation of every stage: the HIP kernels in this
library. Nothing here falls back to another code path: a missing library, a
CPU tensor or an ABI error raises.
"""

from __future__ import annotations

import contextlib
import ctypes
import os
import pathlib
import threading

import torch
from torch.utils._device import DeviceContext

# The in-tree build; CAB_HIP_LIB names another build of the same library (the
# host-sanitized one that tests/test_host_sanitizers.py runs the ABI checks on).
LIB_PATH = pathlib.Path(os.environ.get("CAB_HIP_LIB") or
                        pathlib.Path(__file__).resolve().with_name("libcab_hip.so"))
ABI_VERSION = 11

CAB_OK, CAB_EINVAL, CAB_EDTYPE, CAB_ESHAPE, CAB_EWORKSPACE, CAB_EHIP = range(6)
CAB_F32, CAB_F16, CAB_BF16 = 0, 1, 2
NORMALIZATIONS = {"none": 0, "minmax": 1}
FORMULAS = {"additive": 0, "multiplicative": 1, "augmented": 2}

# Every symbol the header declares, with its ctypes signature.
_i64 = ctypes.c_int64
_i32 = ctypes.c_int32
_ptr = ctypes.c_void_p
_f32 = ctypes.c_float
_i64x4 = ctypes.POINTER(ctypes.c_int64)
SIGNATURES = {
    "cab_abi_version": (ctypes.c_int, []),
    "cab_last_error": (ctypes.c_char_p, []),
    "cab_coarsen_maxl2": (ctypes.c_int, [_ptr, _ptr, ctypes.c_int, _i64, _i64, _i64, _i64,
                                         _i64x4, _i64x4, _i32, _ptr, _ptr, _ptr, _ptr, _ptr]),
    "cab_block_frc_workspace_bytes": (ctypes.c_size_t, [_i64, _i64, _i64, _i64, ctypes.c_int,
                                                        ctypes.c_int]),
    "cab_block_frc": (ctypes.c_int, [_ptr, _ptr, ctypes.c_int, _i64, _i64, _i64, _i64, _f32, _f32,
                                     _f32, ctypes.c_int, ctypes.c_int, _ptr, _ptr, _ptr, _ptr,
                                     ctypes.c_size_t, _ptr]),
    "cab_block_topk": (ctypes.c_int, [_ptr, _i64, _i64, _i64, _i32, ctypes.c_int, ctypes.c_int,
                                      ctypes.c_int, _ptr, _ptr, _ptr, _ptr]),
    "cab_block_topk_hybrid": (ctypes.c_int, [_ptr, _ptr, _i64, _i64, _i64, _i32, _i32, ctypes.c_int,
                                             ctypes.c_int, ctypes.c_int, _ptr, _ptr, _ptr, _ptr]),
    "cab_block_sparse_attn_workspace_bytes": (ctypes.c_size_t, [ctypes.c_int, _i64, _i64, _i64, _i64,
                                                                _i32]),
    "cab_block_sparse_attn_workspace_bytes_k": (ctypes.c_size_t, [ctypes.c_int, _i64, _i64, _i64,
                                                                  _i64, _i32, _i32]),
    "cab_block_sparse_attn_fwd": (ctypes.c_int, [_ptr, _ptr, _ptr, ctypes.c_int, _i64, _i64, _i64,
                                                 _i64, _i64x4, _i64x4, _i64x4, _i64x4, _i32, _ptr,
                                                 _ptr, _i32, _f32, ctypes.c_int, _ptr, _ptr, _ptr,
                                                 ctypes.c_size_t, _ptr]),
    "cab_block_sparse_attn_pack_v": (ctypes.c_int, [_ptr, ctypes.c_int, _i64, _i64, _i64, _i64,
                                                    _i64x4, _i32, _ptr, ctypes.c_size_t, _ptr]),
    "cab_block_sparse_attn_fwd_packed": (ctypes.c_int, [_ptr, _ptr, _ptr, ctypes.c_int, _i64, _i64,
                                                        _i64, _i64, _i64x4, _i64x4, _i64x4, _i32,
                                                        _ptr, _ptr, _i32, _f32, ctypes.c_int, _ptr,
                                                        _ptr, ctypes.c_size_t, _ptr]),
    "cab_flash_attn_workspace_bytes": (ctypes.c_size_t, [ctypes.c_int, _i64, _i64, _i64, _i64]),
    "cab_flash_attn_fwd": (ctypes.c_int, [_ptr, _ptr, _ptr, ctypes.c_int, _i64, _i64, _i64, _i64,
                                          _i64, _i64, _i64x4, _i64x4, _i64x4, _i64x4, _f32,
                                          ctypes.c_int, _ptr, _ptr, _ptr, ctypes.c_size_t, _ptr]),
    "cab_attn_key_scores": (ctypes.c_int, [_ptr, _ptr, _ptr, ctypes.c_int, _i64, _i64, _i64, _i64,
                                           _i64, _i64, _i64x4, _i64x4, _f32, ctypes.c_int, _ptr,
                                           _i64x4, ctypes.c_int, _ptr]),
    "cab_flash_attn_scores_workspace_bytes": (ctypes.c_size_t, [ctypes.c_int, _i64, _i64, _i64, _i64,
                                                                _i64, _i64, _i64x4, _i64x4,
                                                                ctypes.c_int]),
    "cab_flash_attn_scores_fwd": (ctypes.c_int, [_ptr, _ptr, _ptr, ctypes.c_int, _i64, _i64, _i64,
                                                 _i64, _i64, _i64, _i64x4, _i64x4, _i64x4, _i64x4,
                                                 _f32, ctypes.c_int, _ptr, _ptr, _ptr, _i64x4, _i64,
                                                 _ptr, _i64x4, _ptr, ctypes.c_size_t, _ptr]),
    "cab_evict_select_workspace_bytes": (ctypes.c_size_t, [_i64]),
    "cab_evict_select": (ctypes.c_int, [_ptr, _i64, _ptr, _i64, _i32, _i32, _i32, ctypes.c_int,
                                        ctypes.c_int, _ptr, _ptr, _ptr, _ptr, ctypes.c_size_t,
                                        _ptr]),
    "cab_evict_select_noalloc": (ctypes.c_int, [_ptr, _i64, _ptr, _i64, _i32, _i32, _i32,
                                                ctypes.c_int, ctypes.c_int, _ptr, _ptr, _ptr,
                                                _ptr]),
    "cab_evict_connectivity": (ctypes.c_int, [_ptr, _i64, _i64, _ptr, _ptr, _ptr]),
    "cab_kv_gather": (ctypes.c_int, [ctypes.POINTER(_ptr), ctypes.POINTER(_ptr), _i32, _i64, _i64,
                                     _i64, _i64, _i64x4, _i64x4, _ptr, _i64, _ptr]),
    "cab_kv_append": (ctypes.c_int, [_ptr, _ptr, _ptr, _ptr, _i32, _i64, _i64, _i64, _i64, _i64x4,
                                     _i64x4, _i64x4, _i64, _ptr]),
    "cab_key_sums": (ctypes.c_int, [_ptr, ctypes.c_int, _i64, _i64, _i64, _i64, _i64x4, _ptr, _i64,
                                    _ptr, _ptr]),
    "cab_token_frc": (ctypes.c_int, [_ptr, ctypes.c_int, _i64, _i64, _ptr, _ptr, _ptr, _ptr]),
    "cab_attention_symmetrize": (ctypes.c_int, [_ptr, ctypes.c_int, _i64, _i64, _i64, _i64, _i64x4,
                                                _ptr, _i64, _ptr]),
    "cab_token_frc_keys_workspace_bytes": (ctypes.c_size_t, [_i64, _i64]),
    "cab_token_frc_from_keys": (ctypes.c_int, [_ptr, ctypes.c_int, _i64, _i64, _i64, _i64, _i64x4,
                                               _ptr, _ptr, _ptr, _ptr, _ptr, ctypes.c_size_t,
                                               _ptr]),
}

_lock = threading.Lock()
_lib = None


class CabError(RuntimeError):
    """A libcab_hip call failed (status code + message from cab_last_error)."""

    def __init__(self, fn: str, status: int, message: str):
        super().__init__(f"{fn} failed with status {status}: {message}")
        self.status = status


def load() -> ctypes.CDLL:
    """Open libcab_hip.so once (torch must be imported first: the library binds
    to the HIP runtime torch already loaded)."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not LIB_PATH.exists():
                raise RuntimeError(
                    f"{LIB_PATH} is missing: build it with __graft_entry__.build() "
                    "(hipcc, gfx950). There is no fallback implementation.")
            lib = ctypes.CDLL(str(LIB_PATH))
            for name, (res, args) in SIGNATURES.items():
                fn = getattr(lib, name)
                fn.restype = res
                fn.argtypes = args
            ver = lib.cab_abi_version()
            if ver != ABI_VERSION:
                raise RuntimeError(f"libcab_hip ABI version {ver}, expected {ABI_VERSION}")
            _lib = lib
    return _lib


def check(fn: str, status: int) -> None:
    if status != CAB_OK:
        msg = load().cab_last_error().decode(errors="replace")
        if status in (CAB_EINVAL, CAB_EDTYPE, CAB_ESHAPE, CAB_EWORKSPACE):
            raise ValueError(f"{fn}: {msg} (status {status})")
        raise CabError(fn, status, msg)


_DTYPE_CODES = {torch.float32: CAB_F32, torch.float16: CAB_F16, torch.bfloat16: CAB_BF16}


def dtype_code(t: torch.Tensor) -> int:
    code = _DTYPE_CODES.get(t.dtype)
    if code is None:
        raise TypeError(f"unsupported dtype {t.dtype}; expected float32, float16 or bfloat16")
    return code


def require_device(*tensors: torch.Tensor) -> torch.device:
    dev = None
    for t in tensors:
        if not isinstance(t, torch.Tensor):
            raise TypeError(f"expected a torch.Tensor, got {type(t).__name__}")
        if not t.is_cuda:
            raise RuntimeError(
                "CAB-Attention kernels run on the GPU only (HIP, gfx950); got a tensor on "
                f"{t.device}. Move inputs to a cuda device.")
        if dev is None:
            dev = t.device
        elif t.device != dev:
            raise RuntimeError(f"tensors on different devices: {dev} and {t.device}")
    return dev


I64x4 = ctypes.c_int64 * 4


def strides4(t: torch.Tensor):
    return I64x4(*t.stride())


def rows_aligned(t: torch.Tensor) -> bool:
    """Last dim contiguous and rows starting on 16-byte boundaries (what the
    kernels' vector loads need)."""
    st = t.stride()
    if st[-1] != 1 or t.data_ptr() & 15:
        return False
    bits = 0
    for s in st[:-1]:
        bits |= s
    return (bits * t.element_size()) & 15 == 0


def aligned_rows(t: torch.Tensor) -> torch.Tensor:
    """Return ``t`` or a contiguous copy with :func:`rows_aligned` rows."""
    if rows_aligned(t):
        return t
    t = t.contiguous()
    return t if rows_aligned(t) else t.clone()


_PLAIN = (torch.Tensor, torch.nn.Parameter)
# Looked up once: a decode step asks addressable() per layer.
_is_compiling = torch.compiler.is_compiling
_is_tracing = torch._C._is_tracing
_interpreter = torch._C._functorch.peek_interpreter_stack
_dispatch_modes = torch._C._len_torch_dispatch_stack
_function_modes = torch._C._len_torch_function_stack
_forward_ad = torch.autograd.forward_ad


def addressable(*tensors: torch.Tensor) -> bool:
    """Whether a kernel may stand in for torch ops on ``tensors``: plain tensors
    whose memory holds their values (no negative bit), with no transform (vmap,
    forward-mode, tracing) and no mode that has to see the ops."""
    if _is_compiling():
        return False
    for t in tensors:
        if type(t) not in _PLAIN or t.is_neg():
            return False
    return (_interpreter() is None and _forward_ad._current_level < 0 and not _is_tracing()
            and not _dispatch_modes() and (not _function_modes() or _only_device_modes()))


def _only_device_modes() -> bool:
    """Whether the active function modes are default devices alone, which no op on
    existing tensors asks."""
    return all(type(m) is DeviceContext
               for m in torch.overrides._get_current_function_mode_stack())


def closed(t: torch.Tensor) -> bool:
    """Whether torch refuses in-place writes into ``t`` here (an inference tensor
    outside inference mode)."""
    return t.is_inference() and not torch.is_inference_mode_enabled()


def wrote(*tensors: torch.Tensor) -> None:
    """Tells autograd of a kernel's writes into ``tensors``, as torch's in-place ops
    do: a backward pass that saved them raises instead of reading new values."""
    torch._C._increment_version(tensors)


_SAME_DEVICE = contextlib.nullcontext()


def on_device(device: torch.device):
    """Context in which ``device`` is current (nothing to switch if it already
    is, the usual case: a decode step's launches cost as much as their kernels)."""
    if device.index is None or device.index == torch.cuda.current_device():
        return _SAME_DEVICE
    return torch.cuda.device(device)


raw_stream = torch._C._cuda_getCurrentRawStream  # of a device index


def stream_ptr(device: torch.device) -> int:
    index = torch.cuda.current_device() if device.index is None else device.index
    return raw_stream(index)


def ptr(t):
    return None if t is None else t.data_ptr()
