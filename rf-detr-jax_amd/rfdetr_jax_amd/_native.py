"""ctypes binding of the HIP library's C ABI (include/msda.h).

There is no CPU fallback: if the library is missing, :func:`lib` raises, and every op that
needs it fails loudly.
"""

from __future__ import annotations

import contextlib
import ctypes
import importlib.util
import os
import threading
import warnings

import torch

from .build import BINDING_PATH, LIB_PATH

DTYPE_F32 = 0
DTYPE_BF16 = 1

OK = 0
ERR_INVALID_ARGUMENT = -1
ERR_UNSUPPORTED = -2
ERR_LAUNCH = -3
ERR_DEVICE = -4

#: Every function include/msda.h declares, with its ctypes signature.
_I = ctypes.c_int
_P = ctypes.c_void_p
_I32P = ctypes.POINTER(ctypes.c_int32)
_I64 = ctypes.c_int64
_DIMS = [_I] * 6 + [_I32P, _I32P, _I64]  # batch .. n_points, spatial_shapes, level_start_index, len_value
SIGNATURES = {
    "msda_version": ([], ctypes.c_char_p),
    "msda_last_error": ([], ctypes.c_char_p),
    "msda_set_tuning": ([ctypes.c_char_p, ctypes.c_char_p], _I),
    "msda_fwd": ([_P, _I, _P, _P, _P, _I] + _DIMS + [_P], _I),
    "msda_fwd_sampler": ([_P, _I, _P, _P, _P, _I, _I] + _DIMS + [_P], _I),
    "msda_bwd_workspace_size": (list(_DIMS), _I64),
    "msda_bwd": ([_P, _I, _P, _P, _P, _I, _P, _P, _P] + _DIMS + [_P, _I64, _P], _I),
    "msda_bwd_sampler": ([_P, _I, _P, _P, _P, _I, _P, _P, _P, _I] + _DIMS + [_P, _I64, _P], _I),
    "msda_bwd_noalloc": ([_P, _I, _P, _P, _P, _I, _P, _P, _P] + _DIMS + [_P], _I),
    "msda_fused_fwd": ([_P, _I, _P, _I, _P, _P, _P, _I] + _DIMS + [_P], _I),
    "msda_fused_bwd_workspace_size": ([_I] * 7 + [_I32P, _I32P, _I64], _I64),
    "msda_fused_bwd": ([_P, _I, _P, _I, _P, _P, _P, _I, _P, _P, _P, _P] + _DIMS + [_P, _I64, _P], _I),
    "msda_grid_sample_fwd": ([_P, _I, _P, _I, _P] + [_I] * 7 + [_P], _I),
    "msda_grid_sample_bwd": ([_P, _I, _P, _I, _P, _P, _P] + [_I] * 7 + [_P], _I),
    "msda_value_proj_fwd": ([_P, _I, _P, _P, _P, _P] + [_I] * 5 + [_P], _I),
    "msda_value_proj_bwd_workspace_size": ([_I] * 5, _I64),
    "msda_value_proj_bwd": ([_P, _I, _P, _P, _P, _P, _P, _P] + [_I] * 5 + [_P, _I64, _P], _I),
    "msda_attention_fwd": ([_P, _P, _P, _I, _P, _P] + [_I] * 5 + [_P, _P, _P], _I),
    "msda_attention_bwd": ([_P, _P, _P, _P, _P, _P, _I, _P, _P, _P] + [_I] * 5 + [_P, _P, _P], _I),
    "msda_attention_fwd_dropout": ([_P, _P, _P, _I, _P, _P] + [_I] * 5 + [_P, _P, ctypes.c_float, ctypes.c_uint64, _P], _I),
    "msda_attention_bwd_dropout": ([_P, _P, _P, _P, _P, _P, _I, _P, _P, _P] + [_I] * 5
                                   + [_P, _P, ctypes.c_float, ctypes.c_uint64, _P], _I),
    "msda_attention_dropout_keep": ([_I] * 4 + [ctypes.c_float, ctypes.c_uint64, _P, _P], _I),
    # include/msda_probe.h
    "msda_probe_lds_read": ([_P, _I, _I, _P], _I),
    "msda_probe_lds_read_bytes": ([_I, _I], _I64),
    "msda_probe_lds_atomic": ([_P, _I, _I, _P], _I),
    "msda_probe_lds_atomic_f32": ([_P, _I, _I, _P], _I),
    "msda_probe_lds_atomic_ops": ([_I, _I], _I64),
}

GRID_COORDS = 0
GRID_UNIT_POINTS = 1
PADDING = {"zeros": 0, "border": 1}
SAMPLE_BILINEAR = 0
SAMPLE_NEAREST = 1

_lock = threading.Lock()
_lib = None
_binding = None


class MsdaError(RuntimeError):
    """A failed library call; ``code`` is the MSDA_ERR_* status."""

    def __init__(self, code: int, message: str):
        super().__init__(f"msda error {code}: {message}")
        self.code = code


def _library_path() -> str:
    return os.environ.get("MSDA_LIBRARY", LIB_PATH)


def lib(path: str | None = None) -> ctypes.CDLL:
    """Load (once) and return the HIP library."""
    global _lib
    if _lib is not None and path is None:
        return _lib
    with _lock:
        if _lib is not None and path is None:
            return _lib
        target = path or _library_path()
        if not os.path.exists(target):
            raise RuntimeError(
                f"HIP library not found at {target}; build it with __graft_entry__.build() "
                "(hipcc --offload-arch=gfx950). There is no CPU fallback."
            )
        handle = ctypes.CDLL(target)
        for name, (argtypes, restype) in SIGNATURES.items():
            fn = getattr(handle, name)
            fn.argtypes = argtypes
            fn.restype = restype
        if path is None:
            _lib = handle
        return handle


class _NoBinding:
    """Leaves every call to the Python autograd functions."""

    core = fused = value_proj = grid_sample = attention = staticmethod(lambda *args: None)


def binding():
    """Load (once) and return the torch binding: the differentiable ops as C++ autograd functions over
    the library's C ABI, each returning None for a call that the Python path has to take. Without the
    library the Python path reports what is missing; without the binding, which only saves host time,
    it takes every call."""
    global _binding
    if _binding is not None:
        return _binding
    if _lib is None and not os.path.exists(_library_path()):
        return _NoBinding
    handle = lib()
    with _lock:
        if _binding is not None:
            return _binding
        try:
            spec = importlib.util.spec_from_file_location("rfdetr_jax_amd._torch_binding", BINDING_PATH)
            module = importlib.util.module_from_spec(spec)
            spec.loader.exec_module(module)
        except ImportError as e:  # not built, or built against another torch
            warnings.warn(f"the torch binding at {BINDING_PATH} does not load ({e}); every call takes the slower Python path. "
                          "Build it with __graft_entry__.build().", RuntimeWarning, stacklevel=3)
            _binding = _NoBinding
            return _binding
        address = {name: ctypes.cast(getattr(handle, name), ctypes.c_void_p).value for name in SIGNATURES}
        module.bind(address, check, torch.nn.Parameter)
        _binding = module
        return _binding


def check(rc: int) -> None:
    if rc != OK:
        msg = lib().msda_last_error().decode("utf-8", "replace")
        raise MsdaError(rc, msg)


def workspace(nbytes: int, device) -> torch.Tensor:
    """Scratch memory of at least ``nbytes`` (16-byte aligned, in whole 16-byte rows); torch's caching
    allocator serves it."""
    return torch.empty((max(1, (nbytes + 15) // 16), 4), dtype=torch.int32, device=device)


@contextlib.contextmanager
def tuning(knobs: dict):
    """Override launch-tuning knobs (``{"MSDA_BWD_BANDS": 7, ...}``) for the duration of a block;
    the library reads them from the environment only once, so this is how a process switches
    launch variants (benchmarks, tests)."""
    set_ = []
    try:
        for name, value in knobs.items():
            check(lib().msda_set_tuning(name.encode(), str(value).encode()))
            set_.append(name)
        yield
    finally:
        for name in set_:
            lib().msda_set_tuning(name.encode(), None)
