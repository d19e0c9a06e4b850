"""ctypes binding of libentropy_engine.so (include/entropy_engine.h).

The library is loaded after torch so that it binds to the HIP runtime torch
already has in the process (both carry the soname libamdhip64.so.7): one
runtime, so torch's streams and device pointers are valid handles here.
There is no CPU fallback: without the built library or without a GPU every
entry point raises.
"""
from __future__ import annotations

import ctypes
import os
import threading

import torch

PKG_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB_DIR = os.environ.get("EE_LIB_DIR", os.path.join(PKG_ROOT, "lib"))
LIB_PATH = os.path.join(LIB_DIR, "libentropy_engine.so")

# status codes (ee_status)
EE_OK = 0
EE_ERR_INVALID_ARG = -1
EE_ERR_IO = -2
EE_ERR_META = -3
EE_ERR_HIP = -4
EE_ERR_UNSUPPORTED = -5
EE_ERR_NOT_FOUND = -6
STATUS_NAMES = {0: "EE_OK", -1: "EE_ERR_INVALID_ARG", -2: "EE_ERR_IO", -3: "EE_ERR_META", -4: "EE_ERR_HIP",
                -5: "EE_ERR_UNSUPPORTED", -6: "EE_ERR_NOT_FOUND"}

# quantiser modes / GEMM kinds / tiers
EE_QUANT_I8_DISPATCH, EE_QUANT_I8_ENGINE, EE_QUANT_F8_ROW, EE_QUANT_F8_TENSOR = 0, 1, 2, 3
EE_TENSOR_WS_FLOATS = 1024
EE_NOALLOC_MAX_ROWS = 16384              # ee_routed_linear_noalloc's workspace limits
EE_NOALLOC_MAX_CODE_BYTES = 32 * 1024 * 1024
EE_GEMM_I8, EE_GEMM_F8, EE_GEMM_F16, EE_GEMM_W8A16 = 0, 1, 2, 3
EE_ROUTED_SWIGLU, EE_ROUTED_PREQUANT = 1, 2    # flags of ee_routed_linear_packed

_p = ctypes.c_void_p
_i32 = ctypes.c_int32
_i64 = ctypes.c_int64
_f64 = ctypes.c_double

SIGNATURES = {
    "ee_last_error": ([], ctypes.c_char_p),
    "ee_abi_version": ([], ctypes.c_int),
    "ee_engine_create": ([ctypes.c_char_p, ctypes.POINTER(_p)], ctypes.c_int),
    "ee_engine_destroy": ([_p], ctypes.c_int),
    "ee_engine_set_option": ([_p, ctypes.c_char_p, _i64], ctypes.c_int),
    "ee_engine_device": ([_p], ctypes.c_int),
    "ee_last_kernel": ([], ctypes.c_char_p),
    "ee_softmax_entropy": ([_p, _p, _p, _p, _i64, _i32, _i64, _i64, _i32, _p, _f64, _f64, _p], ctypes.c_int),
    "ee_quant_act": ([_p, _p, _i64, _i64, _i64, _i32, _p, _i64, _p, _p, _p, _i32, _p], ctypes.c_int),
    "ee_quant_weight_i8": ([_p, _p, _i64, _i64, _i64, _p, _i64, _p, _p], ctypes.c_int),
    "ee_quant_tensor_f8": ([_p, _p, _i64, _i64, _i64, _p, _i64, _p, _p, _p], ctypes.c_int),
    "ee_transpose_i8": ([_p, _p, _i64, _i64, _i64, _p, _i64, _p], ctypes.c_int),
    "ee_pack_b_f8": ([_p, _p, _i64, _i64, _i64, _p, _i64, _p], ctypes.c_int),
    "ee_pack_b_f16": ([_p, _p, _p, _i64, _i64, _i64, _p, _i64, _p], ctypes.c_int),
    "ee_gemm": ([_p, _i32, _p, _i64, _p, _i64, _p, _i64, _p, _p, _i32, _i32, _i32, _p, _p, _p, _i32, _p, _p],
                ctypes.c_int),
    "ee_gemm_swiglu": ([_p, _i32, _p, _i64, _p, _i64, _p, _i64, _p, _p, _i32, _i32, _i32, _p, _p, _p, _i32, _p],
                       ctypes.c_int),
    "ee_routed_linear_swiglu": ([_p, _p, _i64, _i32, _i32, _i32, _p, _p, _p, _p, _p, _p, _p, _i64, _p, _p, _p],
                                ctypes.c_int),
    "ee_routed_linear_packed": ([_p, _p, _i64, _i32, _i32, _i32, _p, _p, _p, _p, _p, _p, _p, _i64, _p, _p, _i32, _p],
                                ctypes.c_int),
    "ee_gemm_small_waves": ([_p, _i32, _i64, _i64, _i64, _i32], ctypes.c_int),
    "ee_interleave_gate_up": ([_p, _p, _i64, _p, _i64, _i64, _i64, _p], ctypes.c_int),
    "ee_route": ([_p, _p, _i64, _f64, _f64, _p, _p, _p, _p], ctypes.c_int),
    "ee_route_heads": ([_p, _p, _i32, _i32, _i32, _f64, _f64, _p, _p, _p, _p], ctypes.c_int),
    "ee_route_tally": ([_p, _p, _p, _i32, _i64, _p, _p], ctypes.c_int),
    "ee_row_mean": ([_p, _p, _i64, _i32, _p, _p], ctypes.c_int),
    "ee_row_copy": ([_p, _p, _i64, _p, _i64, _i64, _i64, _p, _p, _i32, _i32, _p], ctypes.c_int),
    "ee_routed_linear_noalloc": ([_p, _p, _i64, _i32, _i32, _i32, _p, _p, _p, _p, _p, _p, _p, _i64, _p],
                                 ctypes.c_int),
    "ee_routed_linear": ([_p, _p, _i64, _i32, _i32, _i32, _p, _p, _p, _p, _p, _p, _p, _i64, _p, _p, _p],
                         ctypes.c_int),
    "ee_silu_mul": ([_p, _p, _i64, _p, _i64, _i64, _i64, _p], ctypes.c_int),
    "ee_add_rmsnorm": ([_p, _p, _i64, _p, _i64, _p, _p, _i64, _p, _i64, _i64, _i64, ctypes.c_float, _p], ctypes.c_int),
    "ee_add_rmsnorm_route": ([_p, _p, _i64, _p, _i64, _p, _p, _i64, _p, _i64, _i64, _i64, ctypes.c_float, _p, _p, _p,
                              _i64, _p, _p], ctypes.c_int),
    "ee_routed_gemm": ([_p, _p, _i64, _i32, _i32, _i32, _p, _p, _p, _p, _p, _p, _p, _i64, _p, _p, _p], ctypes.c_int),
    "ee_routed_gemm_swiglu": ([_p, _p, _i64, _i32, _i32, _i32, _p, _p, _p, _p, _p, _p, _p, _i64, _p, _p, _p],
                              ctypes.c_int),
    "ee_qkv_rope": ([_p, _p, _i64, _p, _p, _p, _p, _p, _i32, _i32, _i32, _i32, _i32, ctypes.c_float, _p],
                    ctypes.c_int),
    "ee_qkv_rope_vt": ([_p, _p, _i64, _p, _p, _p, _p, _p, _i32, _i32, _i32, _i32, _i32, ctypes.c_float, _p],
                       ctypes.c_int),
    "ee_attention_causal": ([_p, _p, _p, _p, _p, _i64, _p, _i32, _i32, _i32, _i32, _i32, _p], ctypes.c_int),
    "ee_qkv_rope_vt_pad": ([_p, _p, _i64, _p, _p, _p, _p, _p, _i32, _i32, _i32, _i32, _i32, ctypes.c_float, _p],
                           ctypes.c_int),
    "ee_attention_causal_any": ([_p, _p, _p, _p, _p, _i64, _p, _i32, _i32, _i32, _i32, _i32, _p], ctypes.c_int),
    "ee_mlp_prepare": ([_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _p, _p, _p, _p, _p, _p, _p, _p, _p],
                       ctypes.c_int),
    "ee_mlp_workspace_bytes": ([_i64, _i64, _i64, _i32], _i64),
    "ee_mlp_forward": ([_p, _p, _i64, _i64, _i64, _i64, _p, _p, _p, _p, _p, _p, _p, _p, _f64, _p, _f64, _f64, _p,
                        _i64, _p, _i64, _p], ctypes.c_int),
    "ee_module_engine_create": ([ctypes.c_char_p, ctypes.c_char_p, _i32, _i32, _i32, _i32, ctypes.POINTER(_p)],
                                ctypes.c_int),
    "ee_module_engine_from_metadata": ([ctypes.c_char_p, ctypes.c_char_p, ctypes.c_char_p, ctypes.POINTER(_p)],
                                       ctypes.c_int),
    "ee_module_engine_info": ([_p, ctypes.POINTER(_i32), ctypes.POINTER(_i32), ctypes.POINTER(_i32),
                               ctypes.POINTER(_i32)], ctypes.c_int),
    "ee_module_engine_forward": ([_p, _p, _i64, _p, _i64, _p, _i64, _p, _p, _i32, _i32, _i32, _p], ctypes.c_int),
    "ee_module_engine_destroy": ([_p], ctypes.c_int),
}

_lib = None
_lock = threading.Lock()
_engines: dict[int, int] = {}


class EngineError(RuntimeError):
    """A C-ABI call returned a non-zero ee_status."""

    def __init__(self, status: int, message: str):
        super().__init__(message)
        self.status = status
        self.status_name = STATUS_NAMES.get(status, str(status))


def lib() -> ctypes.CDLL:
    """The loaded C-ABI library (raises if it has not been built)."""
    global _lib
    if _lib is None:
        with _lock:
            if _lib is None:
                if not os.path.exists(LIB_PATH):
                    raise ImportError(
                        f"entropy_engine: native library missing at {LIB_PATH}; "
                        "build it with `python triton-kernels-optimization_amd/build.py`")
                L = ctypes.CDLL(LIB_PATH)
                for name, (args, res) in SIGNATURES.items():
                    fn = getattr(L, name)
                    fn.argtypes = args
                    fn.restype = res
                _lib = L
    return _lib


def check(rc: int) -> None:
    if rc != EE_OK:
        msg = lib().ee_last_error()
        raise EngineError(rc, (msg.decode() if msg else "") or STATUS_NAMES.get(rc, str(rc)))


class _NoSwitch:
    """The context of a call whose device is the current one already."""
    __slots__ = ()

    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_NO_SWITCH = _NoSwitch()
# The current stream's raw handle; through torch.cuda.current_stream() it costs 3 us per call (a Stream object).
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def on_device(dev: torch.device):
    """torch.cuda.device(dev), without its set/restore where dev is current (1.4 us per call)."""
    return _NO_SWITCH if dev.index == torch.cuda.current_device() else torch.cuda.device(dev)


def engine(device=None) -> int:
    """Per-device engine handle (code objects loaded once per device)."""
    if device is None and _engines:                  # (an engine exists: so does a GPU)
        h = _engines.get(torch.cuda.current_device())
        if h is not None:
            return h
    if not torch.cuda.is_available():
        raise RuntimeError("entropy_engine needs a ROCm GPU (gfx950); none is visible")
    dev = torch.cuda.current_device() if device is None else torch.device(device).index
    if dev is None:
        dev = torch.cuda.current_device()
    h = _engines.get(dev)
    if h is None:
        with _lock:
            h = _engines.get(dev)
            if h is None:
                L = lib()
                out = _p()
                with torch.cuda.device(dev):
                    torch.cuda.init()
                    check(L.ee_engine_create(LIB_DIR.encode(), ctypes.byref(out)))
                h = out.value
                _engines[dev] = h
    return h


def stream_handle(device=None) -> int:
    if device is None and _raw_stream is not None:
        return _raw_stream(torch.cuda.current_device())
    return torch.cuda.current_stream(device).cuda_stream


def engine_of(dev: torch.device) -> int:
    """engine(dev) for a tensor's device."""
    return _engines.get(dev.index) or engine(dev)


def stream_of(dev: torch.device) -> int:
    """stream_handle(dev) for a tensor's device."""
    return _raw_stream(dev.index) if _raw_stream is not None else stream_handle(dev)


def ptr(t) -> int | None:
    return None if t is None else t.data_ptr()
