"""ctypes binding of libolmax_hip.so — the C-ABI boundary of the HIP hot path.

The library is built in-tree by :mod:`olmax_amd.build`.  There is deliberately no
fallback: if the shared object is missing, or a call returns a non-zero code, an
exception is raised.
"""
from __future__ import annotations

import ctypes
from ctypes import c_char_p, c_double, c_float, c_int32, c_int64, c_void_p
from pathlib import Path

_LIB_PATH = Path(__file__).resolve().parent / "libolmax_hip.so"
_lib = None


class OlmaxHipError(RuntimeError):
    pass


def lib_path() -> Path:
    return _LIB_PATH


def load() -> ctypes.CDLL:
    """Load (once) and return the shared library; raise if it has not been built."""
    global _lib
    if _lib is None:
        if not _LIB_PATH.exists():
            raise OlmaxHipError(
                f"{_LIB_PATH} not found: build it with `python -m olmax_amd.build` "
                "(there is no CPU or eager fallback for the HIP path)"
            )
        _lib = ctypes.CDLL(str(_LIB_PATH))
        _lib.olmax_last_error_string.restype = c_char_p
        _lib.olmax_abi_version.restype = c_int32
    return _lib


def check(rc: int) -> None:
    if rc != 0:
        msg = load().olmax_last_error_string().decode()
        raise OlmaxHipError(f"libolmax_hip error {rc}: {msg}")


def ptr(t) -> c_void_p:
    """Raw device pointer of a torch tensor (None -> NULL)."""
    return c_void_p(0 if t is None else t.data_ptr())


def stream_ptr() -> c_void_p:
    """Current stream of the current device; the raw handle, without a Stream object around it (0.3 instead of 3 us of
    an 11 us call)."""
    import torch

    return c_void_p(torch._C._cuda_getCurrentRawStream(torch.cuda.current_device()))


i32, i64, f32, f64, vp = c_int32, c_int64, c_float, c_double, c_void_p

# Argument types of the entry points that a program calls once per layer and pass: P pointer, I int32, L int64, F float.
_SIGNATURES = {
    "olmax_gemm_bf16": "PPPPPIIILLLLIII",
    "olmax_rmsnorm_fwd": "PPPPLILLF",
    "olmax_rmsnorm_bwd": "PPPPPPPLILLLLF",
    "olmax_fill_zero": "PPL",
    "olmax_attn_fwd": "PPPPPPIIIIILLLLIF",
    "olmax_attn_bwd": "PPPPPPPPPPPLIIIIILLLLLLLLIF",
}
_typed = {}


def typed(name: str):
    """Entry point `name` with its argument types set, on a handle of its own: it takes plain integers, floats and None, which ctypes
    converts in C (0.1 us an argument less than an object around each)."""
    f = _typed.get(name)
    if f is None:
        load()
        f = getattr(ctypes.CDLL(str(_LIB_PATH)), name)
        f.argtypes = [{"P": vp, "I": i32, "L": i64, "F": f32}[c] for c in _SIGNATURES[name]]
        f.restype = i32
        _typed[name] = f
    return f


def raw_stream() -> int:
    """Current stream of the current device, as an integer."""
    import torch

    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())
