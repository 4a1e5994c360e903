"""ctypes binding of libaxl_attn_hip.so (the C ABI declared in include/axl_attn.h).

The library is the only compute path: if it cannot be loaded every kernel entry raises. There is no
PyTorch or CPU fallback anywhere in this package.
"""

from __future__ import annotations

import ctypes
import os
import struct
from typing import Optional

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libaxl_attn_hip.so")

AXL_BF16, AXL_F32, AXL_F16 = 0, 1, 2
MASK_NONE, MASK_CAUSAL, MASK_SLIDING_WINDOW = 0, 1, 2
DECODE_DETERMINISTIC, DECODE_WORKSPACE_REUSED = 1, 2  # AXL_DECODE_* flags
DECODE_LENGTHS_ARE_POSITIONS, DECODE_LENGTHS_I64 = 4, 8
BWD_DS_WORKSPACE, BWD_F32_NO_PLANES, BWD_NO_SPLIT = 1, 2, 4  # AXL_BWD_* flags
AXL_OK, AXL_ERR_INVALID_ARGUMENT, AXL_ERR_UNSUPPORTED, AXL_ERR_WORKSPACE, AXL_ERR_LAUNCH = 0, -1, -2, -3, -4


ABI_VERSION = 9  # AXL_ATTN_ABI_VERSION of include/axl_attn.h these structures mirror


class AxlError(RuntimeError):
    """A C-ABI call returned a negative status."""

    def __init__(self, code: int, message: str):
        super().__init__(f"[axl status {code}] {message}")
        self.code = code


class AxlStrides(ctypes.Structure):
    _fields_ = [("batch", ctypes.c_int64), ("seq", ctypes.c_int64), ("head", ctypes.c_int64)]


class AxlAttnAux(ctypes.Structure):
    _fields_ = [
        ("bias", ctypes.c_void_p),
        ("bias_batch_stride", ctypes.c_int64), ("bias_head_stride", ctypes.c_int64),
        ("bias_row_stride", ctypes.c_int64),
        ("bias_dtype", ctypes.c_int32), ("dropout_rate", ctypes.c_float),
        ("dropout_mask", ctypes.c_void_p),
        ("drop_batch_stride", ctypes.c_int64), ("drop_head_stride", ctypes.c_int64),
        ("drop_row_stride", ctypes.c_int64),
    ]


class AxlFlashFwdParams(ctypes.Structure):
    _fields_ = [
        ("q", ctypes.c_void_p), ("k", ctypes.c_void_p), ("v", ctypes.c_void_p),
        ("out", ctypes.c_void_p), ("lse", ctypes.c_void_p), ("segment_ids", ctypes.c_void_p),
        ("q_strides", AxlStrides), ("k_strides", AxlStrides), ("v_strides", AxlStrides),
        ("out_strides", AxlStrides),
        ("batch", ctypes.c_int32), ("q_len", ctypes.c_int32), ("kv_len", ctypes.c_int32),
        ("num_q_heads", ctypes.c_int32), ("num_kv_heads", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("dtype", ctypes.c_int32), ("mask_kind", ctypes.c_int32),
        ("sliding_window", ctypes.c_int32), ("q_pos_offset", ctypes.c_int32),
        ("softmax_scale", ctypes.c_float),
        ("logit_sink", ctypes.c_void_p),
        ("aux", AxlAttnAux),
        ("q_pos_offsets", ctypes.c_void_p),
        ("bias_copy", ctypes.c_void_p),
    ]


class AxlFlashChunkParams(ctypes.Structure):
    _fields_ = [
        ("q", ctypes.c_void_p), ("k", ctypes.c_void_p), ("v", ctypes.c_void_p), ("out", ctypes.c_void_p),
        ("q_strides", AxlStrides), ("k_strides", AxlStrides), ("v_strides", AxlStrides),
        ("out_strides", AxlStrides),
        ("batch", ctypes.c_int32), ("q_len", ctypes.c_int32), ("kv_len", ctypes.c_int32),
        ("num_q_heads", ctypes.c_int32), ("num_kv_heads", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("dtype", ctypes.c_int32), ("mask_kind", ctypes.c_int32),
        ("sliding_window", ctypes.c_int32),
        ("softmax_scale", ctypes.c_float),
        ("logit_sink", ctypes.c_void_p), ("positions", ctypes.c_void_p),
        ("pos_batch_stride", ctypes.c_int64), ("pos_row_stride", ctypes.c_int64),
        ("pos_is_i64", ctypes.c_int32),
        ("workspace", ctypes.c_void_p), ("workspace_bytes", ctypes.c_size_t),
    ]


class AxlFlashBwdParams(ctypes.Structure):
    _fields_ = [
        ("q", ctypes.c_void_p), ("k", ctypes.c_void_p), ("v", ctypes.c_void_p),
        ("out", ctypes.c_void_p), ("d_out", ctypes.c_void_p), ("lse", ctypes.c_void_p),
        ("dq", ctypes.c_void_p), ("dk", ctypes.c_void_p), ("dv", ctypes.c_void_p),
        ("segment_ids", ctypes.c_void_p),
        ("q_strides", AxlStrides), ("k_strides", AxlStrides), ("v_strides", AxlStrides),
        ("out_strides", AxlStrides), ("d_out_strides", AxlStrides),
        ("dq_strides", AxlStrides), ("dk_strides", AxlStrides), ("dv_strides", AxlStrides),
        ("batch", ctypes.c_int32), ("q_len", ctypes.c_int32), ("kv_len", ctypes.c_int32),
        ("num_q_heads", ctypes.c_int32), ("num_kv_heads", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("dtype", ctypes.c_int32), ("mask_kind", ctypes.c_int32),
        ("sliding_window", ctypes.c_int32), ("q_pos_offset", ctypes.c_int32),
        ("softmax_scale", ctypes.c_float),
        ("workspace", ctypes.c_void_p), ("workspace_bytes", ctypes.c_size_t),
        ("logit_sink", ctypes.c_void_p), ("d_logit_sink", ctypes.c_void_p),
        ("aux", AxlAttnAux),
        ("flags", ctypes.c_int32),
    ]


class AxlDecodeBias(ctypes.Structure):
    _fields_ = [
        ("bias", ctypes.c_void_p), ("batch_stride", ctypes.c_int64), ("head_stride", ctypes.c_int64),
        ("dtype", ctypes.c_int32),
    ]


class AxlPagedDecodeParams(ctypes.Structure):
    _fields_ = [
        ("q", ctypes.c_void_p), ("k_pages", ctypes.c_void_p), ("v_pages", ctypes.c_void_p),
        ("page_tables", ctypes.c_void_p), ("lengths", ctypes.c_void_p), ("out", ctypes.c_void_p),
        ("batch", ctypes.c_int32), ("num_q_heads", ctypes.c_int32),
        ("num_kv_heads", ctypes.c_int32), ("head_dim", ctypes.c_int32),
        ("num_pages", ctypes.c_int32), ("page_size", ctypes.c_int32),
        ("pages_per_seq", ctypes.c_int32),
        ("dtype", ctypes.c_int32), ("sliding_window", ctypes.c_int32),
        ("softmax_scale", ctypes.c_float),
        ("workspace", ctypes.c_void_p), ("workspace_bytes", ctypes.c_size_t),
        ("flags", ctypes.c_int32),
        ("bias", AxlDecodeBias),
        ("lengths_stride", ctypes.c_int64),
    ]


class AxlDecodeParams(ctypes.Structure):
    _fields_ = [
        ("q", ctypes.c_void_p), ("k", ctypes.c_void_p), ("v", ctypes.c_void_p),
        ("lengths", ctypes.c_void_p), ("out", ctypes.c_void_p),
        ("k_strides", AxlStrides), ("v_strides", AxlStrides),
        ("batch", ctypes.c_int32), ("kv_len", ctypes.c_int32), ("num_q_heads", ctypes.c_int32),
        ("num_kv_heads", ctypes.c_int32), ("head_dim", ctypes.c_int32),
        ("dtype", ctypes.c_int32), ("sliding_window", ctypes.c_int32),
        ("softmax_scale", ctypes.c_float),
        ("workspace", ctypes.c_void_p), ("workspace_bytes", ctypes.c_size_t),
        ("flags", ctypes.c_int32),
        ("bias", AxlDecodeBias),
        ("lengths_stride", ctypes.c_int64),
    ]


class AxlPageInsertParams(ctypes.Structure):
    _fields_ = [
        ("k_pages", ctypes.c_void_p), ("v_pages", ctypes.c_void_p),
        ("k_proj", ctypes.c_void_p), ("v_proj", ctypes.c_void_p),
        ("page_indices", ctypes.c_void_p), ("key_positions", ctypes.c_void_p),
        ("k_proj_batch_stride", ctypes.c_int64), ("k_proj_head_stride", ctypes.c_int64),
        ("v_proj_batch_stride", ctypes.c_int64), ("v_proj_head_stride", ctypes.c_int64),
        ("batch", ctypes.c_int32), ("num_kv_heads", ctypes.c_int32), ("head_dim", ctypes.c_int32),
        ("num_pages", ctypes.c_int32), ("page_size", ctypes.c_int32), ("pages_per_seq", ctypes.c_int32),
        ("dtype", ctypes.c_int32), ("broadcast_positions", ctypes.c_int32),
    ]


def _packer(cls):
    """fill(*values) -> an instance of the parameter block `cls`, its fields in order and nested blocks flat.

    One `struct.pack` instead of a ctypes assignment per field (24 fields by keyword and four nested blocks took 8 us,
    this 1 us); None is not a pointer here, 0 is."""
    codes = {ctypes.c_void_p: "P", ctypes.c_int64: "q", ctypes.c_int32: "i", ctypes.c_float: "f", ctypes.c_size_t: "N"}

    def layout(c):
        inner = "".join(layout(t) if issubclass(t, ctypes.Structure) else codes[t] for _, t in c._fields_)
        return f"0P{inner}0P"   # every block starts and ends on a pointer's alignment

    packed = struct.Struct("@" + layout(cls))
    assert packed.size == ctypes.sizeof(cls) and ctypes.alignment(cls) == ctypes.alignment(ctypes.c_void_p)
    pack, view = packed.pack, cls.from_buffer
    return lambda *values: view(bytearray(pack(*values)))


fill_flash_fwd, fill_flash_chunk, fill_flash_bwd, fill_paged_decode, fill_decode, fill_page_insert = map(_packer, (
    AxlFlashFwdParams, AxlFlashChunkParams, AxlFlashBwdParams, AxlPagedDecodeParams, AxlDecodeParams, AxlPageInsertParams))


def int32(x) -> int:
    """`x` as the parameter blocks hold it."""
    x = int(x)
    return x if -0x80000000 <= x <= 0x7fffffff else ctypes.c_int32(x).value


def float32(x) -> float:
    """`x` as the parameter blocks hold it: past the type's range infinite, where `struct` would raise."""
    x = float(x)
    return x if -3.4e38 < x < 3.4e38 else ctypes.c_float(x).value


EXPORTED_SYMBOLS = (
    "axl_flash_fwd",
    "axl_flash_chunk",
    "axl_flash_chunk_workspace_bytes",
    "axl_flash_bwd",
    "axl_flash_bwd_phases",
    "axl_flash_bwd_workspace_bytes",
    "axl_paged_decode",
    "axl_paged_decode_workspace_bytes",
    "axl_paged_decode_static",
    "axl_decode",
    "axl_decode_workspace_bytes",
    "axl_paged_kv_insert",
    "axl_last_error",
    "axl_abi_version",
)

_lib: Optional[ctypes.CDLL] = None


def load() -> ctypes.CDLL:
    """Loads the HIP library, or raises: there is nothing to fall back to."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            f"{LIB_PATH} is missing. Build it with `make -C axlearn_amd/csrc` (needs hipcc); "
            "axlearn_amd has no non-HIP execution path."
        )
    lib = ctypes.CDLL(LIB_PATH)
    lib.axl_last_error.restype = ctypes.c_char_p
    lib.axl_abi_version.restype = ctypes.c_int
    if lib.axl_abi_version() != ABI_VERSION:
        raise RuntimeError(
            f"{LIB_PATH} has ABI version {lib.axl_abi_version()}, this binding expects {ABI_VERSION}: "
            "rebuild it with `make -C axlearn_amd/csrc`."
        )
    for name, ptype in (
        ("axl_flash_fwd", AxlFlashFwdParams),
        ("axl_flash_chunk", AxlFlashChunkParams),
        ("axl_flash_bwd", AxlFlashBwdParams),
        ("axl_paged_decode", AxlPagedDecodeParams),
        ("axl_paged_decode_static", AxlPagedDecodeParams),
        ("axl_decode", AxlDecodeParams),
        ("axl_paged_kv_insert", AxlPageInsertParams),
    ):
        fn = getattr(lib, name)
        fn.restype = ctypes.c_int
        fn.argtypes = [ctypes.POINTER(ptype), ctypes.c_void_p]
    lib.axl_flash_bwd_phases.restype = ctypes.c_int
    lib.axl_flash_bwd_phases.argtypes = [ctypes.POINTER(AxlFlashBwdParams), ctypes.c_int, ctypes.c_void_p]
    for name, ptype in (
        ("axl_flash_chunk_workspace_bytes", AxlFlashChunkParams),
        ("axl_flash_bwd_workspace_bytes", AxlFlashBwdParams),
        ("axl_paged_decode_workspace_bytes", AxlPagedDecodeParams),
        ("axl_decode_workspace_bytes", AxlDecodeParams),
    ):
        fn = getattr(lib, name)
        fn.restype = ctypes.c_size_t
        fn.argtypes = [ctypes.POINTER(ptype)]
    _lib = lib
    return lib


def check(rc: int) -> None:
    if rc != AXL_OK:
        raise AxlError(rc, load().axl_last_error().decode())


def dtype_code(dtype: torch.dtype) -> int:
    if dtype == torch.bfloat16:
        return AXL_BF16
    if dtype == torch.float32:
        return AXL_F32
    if dtype == torch.float16:
        return AXL_F16
    raise AxlError(AXL_ERR_UNSUPPORTED, f"dtype {dtype} (supported: bfloat16, float16, float32)")


def strides4(t: torch.Tensor) -> tuple:
    """Strides of a [batch, seq, heads, head_dim] tensor (an AxlStrides); the last dim must be dense."""
    strides = t.stride()
    if len(strides) != 4 or strides[3] != 1:
        raise AxlError(AXL_ERR_UNSUPPORTED, f"expected a 4-d tensor dense in head_dim, got strides {strides}")
    return strides[:3]


def current_stream_ptr() -> int:
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())  # no Stream object around it


def ptr(t: Optional[torch.Tensor]) -> int:
    return 0 if t is None else t.data_ptr()
