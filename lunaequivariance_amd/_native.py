"""Loader and thin ctypes binding of the C-ABI library ``liblunaeq_amd.so``.

The library is built in-tree by ``lunaequivariance_amd.build.build_library``;
importing this module never compiles anything.  A missing library raises
``RuntimeError`` at first use: there is no CPU fallback for the kernels.
"""

from __future__ import annotations

import ctypes
import os
from pathlib import Path

import torch

PACKAGE_DIR = Path(__file__).resolve().parent
LIBRARY_PATH = PACKAGE_DIR / "liblunaeq_amd.so"
DEFAULT_CACHE_DIR = PACKAGE_DIR / "_kcache"


class PlanInfo(ctypes.Structure):
    _fields_ = [(name, ctypes.c_int32) for name in (
        "dtype_bits", "in1_dim", "in2_dim", "out_dim", "weight_numel", "l0_dim",
        "num_paths", "fwd_needs_zero", "bwd_gx_needs_zero", "num_fwd_launches", "gy_parts",
    )]


# Exported symbols and their prototypes: (restype, argtypes).
_VP, _I64, _I32P = ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p
PROTOTYPES = {
    "luna_last_error": (ctypes.c_char_p, []),
    "luna_version": (ctypes.c_char_p, []),
    "luna_device_count": (ctypes.c_int, []),
    "luna_uvu_plan_create": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_char_p, ctypes.POINTER(_VP)]),
    "luna_uvu_plan_create_ex": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_char_p, ctypes.c_int, ctypes.POINTER(_VP)]),
    "luna_uvu_plan_destroy": (ctypes.c_int, [_VP]),
    "luna_uvu_plan_info": (ctypes.c_int, [_VP, ctypes.POINTER(PlanInfo)]),
    "luna_uvu_plan_precompile": (ctypes.c_int, [_VP]),
    "luna_uvu_plan_precompile_all": (ctypes.c_int, [_VP]),
    "luna_uvu_conv_fwd": (ctypes.c_int, [_VP] + [_VP] * 4 + [_I32P] * 3 + [_VP, _VP, _I64, _I64, _VP]),
    "luna_uvu_conv_bwd_workspace": (ctypes.c_int, [_VP, _I64, _I64, ctypes.POINTER(ctypes.c_size_t)]),
    "luna_uvu_conv_bwd": (ctypes.c_int, [_VP] + [_VP] * 6 + [_I32P] * 5 + [_VP] * 5
                          + [ctypes.c_size_t, _I64, _I64, _VP]),
    "luna_uvu_conv_bwd_noalloc_limit": (ctypes.c_size_t, []),
    "luna_uvu_conv_bwd_noalloc": (ctypes.c_int, [_VP] + [_VP] * 6 + [_I32P] * 5 + [_VP] * 4 + [_I64, _I64, _VP]),
    "luna_uvu_rows_fwd": (ctypes.c_int, [_VP] * 4 + [ctypes.c_int, _VP, _I64, _VP]),
    "luna_uvu_rows_bwd_workspace": (ctypes.c_int, [_VP, ctypes.c_int, _I64, ctypes.POINTER(ctypes.c_size_t)]),
    "luna_uvu_rows_bwd": (ctypes.c_int, [_VP] * 4 + [ctypes.c_int] + [_VP] * 5 + [ctypes.c_size_t, _I64, _VP]),
    "luna_uvw_plan_create": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_char_p, ctypes.POINTER(_VP)]),
    "luna_uvw_plan_destroy": (ctypes.c_int, [_VP]),
    "luna_uvw_plan_needs_zero": (ctypes.c_int, [_VP, ctypes.POINTER(ctypes.c_int32)]),
    "luna_uvw_plan_precompile": (ctypes.c_int, [_VP]),
    "luna_uvw_fwd": (ctypes.c_int, [_VP] * 5 + [_I64, _VP]),
    "luna_uvw_bwd_workspace": (ctypes.c_int, [_VP, _I64, ctypes.POINTER(ctypes.c_size_t)]),
    "luna_uvw_bwd": (ctypes.c_int, [_VP] * 9 + [ctypes.c_size_t, _I64, _VP]),
    "luna_con_plan_create": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_char_p, ctypes.POINTER(_VP)]),
    "luna_con_plan_destroy": (ctypes.c_int, [_VP]),
    "luna_con_plan_precompile": (ctypes.c_int, [_VP]),
    "luna_con_fwd": (ctypes.c_int, [_VP] * 4 + [_I64, _VP]),
    "luna_con_grad_a": (ctypes.c_int, [_VP] * 4 + [_I64, _VP]),
    "luna_con_grad_w_workspace": (ctypes.c_int, [_VP, _I64, ctypes.POINTER(ctypes.c_size_t)]),
    "luna_con_grad_w": (ctypes.c_int, [_VP] * 5 + [ctypes.c_size_t, _I64, _VP]),
    "luna_uuu_plan_create": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_char_p, ctypes.POINTER(_VP)]),
    "luna_uuu_plan_create_ex": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_char_p, ctypes.c_int, ctypes.POINTER(_VP)]),
    "luna_uuu_plan_destroy": (ctypes.c_int, [_VP]),
    "luna_uuu_plan_needs_zero": (ctypes.c_int, [_VP, ctypes.POINTER(ctypes.c_int32)]),
    "luna_uuu_plan_precompile": (ctypes.c_int, [_VP]),
    "luna_uuu_conv_fwd": (ctypes.c_int, [_VP] + [_VP] * 4 + [_I32P] * 3 + [_VP, _VP, _I64, _I64, _VP]),
    "luna_uuu_conv_bwd_workspace": (ctypes.c_int, [_VP, _I64, _I64, ctypes.POINTER(ctypes.c_size_t)]),
    "luna_uuu_conv_bwd": (ctypes.c_int, [_VP] + [_VP] * 6 + [_I32P] * 4 + [_VP] * 5
                          + [ctypes.c_size_t, _I64, _I64, _VP]),
    "luna_placed_alloc": (ctypes.c_int, [ctypes.c_size_t, _VP, ctypes.c_size_t, ctypes.c_size_t, _VP,
                                          ctypes.POINTER(_VP), ctypes.POINTER(ctypes.c_int)]),
    "luna_region_overlap": (ctypes.c_int, [_VP, ctypes.c_size_t, _VP, ctypes.c_size_t, _VP,
                                            ctypes.POINTER(ctypes.c_double)]),
    "luna_placed_free": (ctypes.c_int, [_VP]),
    "luna_graph_bounds": (ctypes.c_int, [_VP, _VP, ctypes.c_int, _I64, _VP, _VP]),
    "luna_graph_workspace": (ctypes.c_int, [_I64, _I64, ctypes.POINTER(ctypes.c_size_t)]),
    "luna_graph_build": (ctypes.c_int, [_VP, _VP, ctypes.c_int, _I64, _I64] + [_VP] * 15
                         + [ctypes.c_size_t, _VP]),
    "luna_graph_scan": (ctypes.c_int, [_VP, _VP, ctypes.c_int, _I64, _I64] + [_VP] * 9 + [ctypes.c_size_t, _VP]),
    "luna_graph_finish": (ctypes.c_int, [_VP] * 3 + [_I64] * 4 + [_VP] * 8 + [ctypes.c_size_t, _VP]),
    "luna_graph_precompile": (ctypes.c_int, [ctypes.c_char_p]),
    "luna_profile_enable": (ctypes.c_int, [ctypes.c_int]),
    "luna_profile_collect": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_size_t,
                                             ctypes.POINTER(ctypes.c_size_t)]),
}

_lib = None


def library_available() -> bool:
    return LIBRARY_PATH.exists()


def lib() -> ctypes.CDLL:
    """The loaded C-ABI library (raises RuntimeError if it was never built)."""
    global _lib
    if _lib is None:
        if not LIBRARY_PATH.exists():
            raise RuntimeError(
                f"{LIBRARY_PATH} is missing: build it with "
                "`python -c 'import lunaequivariance_amd.build as b; b.build_library()'`")
        handle = ctypes.CDLL(str(LIBRARY_PATH))
        for name, (restype, argtypes) in PROTOTYPES.items():
            function = getattr(handle, name)
            function.restype = restype
            function.argtypes = argtypes
        _lib = handle
    return _lib


def check(status: int, what: str) -> None:
    if status != 0:
        message = lib().luna_last_error().decode(errors="replace")
        raise RuntimeError(f"{what}: {message}")


def profile_enable(on: bool) -> None:
    check(lib().luna_profile_enable(1 if on else 0), "luna_profile_enable")


def profile_collect() -> dict:
    """{kernel name: (launches, total_ms, min_ms, max_ms)} since the last collect."""
    buffer = ctypes.create_string_buffer(1 << 16)
    needed = ctypes.c_size_t()
    check(lib().luna_profile_collect(buffer, len(buffer), ctypes.byref(needed)), "luna_profile_collect")
    result = {}
    for line in buffer.value.decode().splitlines():
        name, count, total, low, high = line.split()
        result[name] = (int(count), float(total), float(low), float(high))
    return result


def cache_dir() -> str:
    return os.environ.get("LUNAEQ_AMD_CACHE", str(DEFAULT_CACHE_DIR))


def stream_of(tensor) -> int:
    """Handle of the current stream of a GPU tensor's device (``torch.cuda.current_stream``
    builds a stream object first, 3 us of the 14 us that a small forward takes)."""
    return torch._C._cuda_getCurrentRawStream(tensor.get_device())


def ptr(tensor) -> int | None:
    """Device address of a tensor, or None for an absent optional tensor."""
    return None if tensor is None else tensor.data_ptr()


__all__ = ["lib", "check", "cache_dir", "ptr", "stream_of", "PlanInfo", "PROTOTYPES", "LIBRARY_PATH",
           "library_available"]
