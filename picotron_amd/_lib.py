"""Binding of ``libpicotron_hip.so`` (C ABI declared in ``include/picotron_hip.h``): ctypes for
raw arguments, and the ``_native`` extension (``csrc/native.cpp``) for whole calls on tensors.

The library is loaded lazily, once per process.  Loading fails loudly with
:class:`HipLibraryUnavailable` (never a silent fallback) when the shared object is missing or
cannot be opened, or when it or the extension was built for another ABI version.  The extension only saves host time: every call
has a ctypes route to the same kernels, taken with a warning when the extension is missing or cannot
be loaded.  This module needs no torch (the extension is bound once torch is there).
"""

from __future__ import annotations

import ctypes
import importlib
import os
import sys
import threading
import warnings
from ctypes import c_double, c_float, c_int, c_int64, c_size_t, c_void_p
from pathlib import Path

LIB_PATH = Path(os.environ.get("PICOTRON_HIP_LIB", Path(__file__).with_name("libpicotron_hip.so")))

ABI_VERSION = 4

PT_FLOAT32 = 0
PT_FLOAT16 = 1
PT_BFLOAT16 = 2

PT_OK = 0
PT_EINVAL = 1
PT_EUNSUPPORTED = 2
PT_ELAUNCH = 3
PT_EDEVICE = 4

_c_int64_p = ctypes.POINTER(c_int64)
_c_float_p = ctypes.POINTER(c_float)

# name -> (restype, argtypes); mirrors include/picotron_hip.h one to one.
SIGNATURES: dict[str, tuple[object, list[object]]] = {
    "pt_abi_version": (c_int, []),
    "pt_last_error": (ctypes.c_char_p, []),
    "pt_device_supported": (c_int, [c_int]),
    "pt_rmsnorm_fwd": (
        c_int,
        [c_void_p, c_int64, c_void_p, c_void_p, c_int64, c_void_p, c_int64, c_int64, c_float,
         c_int, c_int, c_void_p],
    ),
    "pt_rmsnorm_bwd_workspace_bytes": (c_size_t, [c_int64, c_int64, c_int]),
    "pt_rmsnorm_bwd": (
        c_int,
        [c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_int64, c_void_p,
         c_void_p, c_size_t, c_int64, c_int64, c_int, c_int, c_void_p],
    ),
    "pt_rmsnorm_bwd_noalloc": (
        c_int,
        [c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_int64, c_void_p,
         c_int64, c_int64, c_int, c_int, c_void_p],
    ),
    "pt_residual_rmsnorm_fwd": (
        c_int,
        [c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p, c_int64, c_void_p, c_int64,
         c_void_p, c_int64, c_int64, c_float, c_int, c_int, c_void_p],
    ),
    "pt_residual_rmsnorm_bwd": (
        c_int,
        [c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p, c_void_p,
         c_int64, c_void_p, c_void_p, c_size_t, c_int64, c_int64, c_int, c_int, c_void_p],
    ),
    "pt_swiglu_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_int64, c_int, c_void_p]),
    "pt_swiglu_bwd": (
        c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int, c_void_p]
    ),
    "pt_rope": (
        c_int,
        [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_void_p,
         c_int64, c_int, c_int, c_int, c_void_p],
    ),
    "pt_cross_entropy_workspace_bytes": (c_size_t, [c_int64]),
    "pt_cross_entropy": (
        c_int,
        [c_void_p, c_int64, c_int64, c_int64, c_int64, c_int64, c_void_p, c_int64, c_int64,
         c_int64, c_void_p, c_int, c_void_p, c_int64, c_int64, c_void_p, c_size_t, c_int,
         c_void_p],
    ),
    "pt_cross_entropy_status": (c_void_p, [c_void_p]),
    "pt_cross_entropy_scale_grad": (
        c_int,
        [c_void_p, c_int64, c_int64, c_int64, c_int64, c_int64, c_void_p, c_int64, c_int64,
         c_int64, c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_int, c_void_p],
    ),
    "pt_cross_entropy_shifted": (
        c_int,
        [c_void_p, c_int64, c_int64, c_int64, c_int64, c_int64, c_void_p, c_int64, c_int64,
         c_int64, c_void_p, c_int, c_void_p, c_int64, c_int64, c_void_p, c_size_t, c_int,
         c_void_p],
    ),
    "pt_cross_entropy_shifted_scale_grad": (
        c_int,
        [c_void_p, c_int64, c_int64, c_int64, c_int64, c_int64, c_void_p, c_int64, c_int64,
         c_int64, c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_int, c_void_p],
    ),
    "pt_adamw_block_elems": (c_int64, []),
    "pt_adamw_step": (
        c_int,
        [c_void_p, c_int64, c_int64, c_double, c_double, c_double, c_double, c_double, c_double,
         c_void_p],
    ),
    "pt_clip_grad_norm_workspace_bytes": (c_size_t, [c_int64]),
    "pt_clip_grad_norm": (
        c_int,
        [c_void_p, c_int64, c_int64, c_double, c_void_p, c_void_p, c_void_p, c_size_t, c_void_p],
    ),
    "pt_adamw_step_scaled": (
        c_int,
        [c_void_p, c_int64, c_int64, c_double, c_double, c_double, c_double, c_double, c_double,
         c_void_p, c_int, c_void_p],
    ),
    "pt_adamw_step_device_step": (
        c_int,
        [c_void_p, c_int64, c_int64, c_void_p, c_double, c_double, c_double, c_double, c_double,
         c_void_p, c_int, c_void_p],
    ),
    "pt_adamw_step_device_step_guarded": (
        c_int,
        [c_void_p, c_int64, c_int64, c_void_p, c_double, c_double, c_double, c_double, c_double,
         c_void_p, c_int, c_void_p, c_void_p, c_void_p],
    ),
    "pt_grad_stats_workspace_bytes": (c_size_t, [c_int64]),
    "pt_grad_stats": (
        c_int,
        [c_void_p, c_int64, c_int64, c_void_p, c_double, c_int, c_void_p, c_void_p, c_void_p,
         c_void_p, c_size_t, c_void_p],
    ),
    "pt_grad_scale": (c_int, [c_void_p, c_int64, c_int64, c_void_p, c_void_p]),
    "pt_copy": (c_int, [c_void_p, c_void_p, c_int64, c_void_p]),
}


class HipLibraryUnavailable(RuntimeError):
    """The HIP kernel library could not be loaded (missing, stale, or wrong ABI)."""


class HipKernelError(RuntimeError):
    """A library entry point rejected its arguments or failed to launch."""

    def __init__(self, fn: str, code: int, message: str) -> None:
        super().__init__(f"{fn} failed (code {code}): {message}")
        self.fn = fn
        self.code = code


_lock = threading.Lock()
_lib: ctypes.CDLL | None = None
# entry point -> native launcher taking tensors; filled with the extension
_launchers: dict[str, object] = {}
native = None  # the extension module, or None: every call goes through ctypes
_native_tried = False
_load_error: str | None = None


def _load() -> ctypes.CDLL:
    global _lib, _load_error
    with _lock:
        if _lib is not None:
            return _lib
        if _load_error is not None:
            raise HipLibraryUnavailable(_load_error)
        if not LIB_PATH.exists():
            _load_error = (
                f"{LIB_PATH} is not built (run `python -m picotron_amd.build` or "
                "`python -c 'import __graft_entry__ as g; g.build()'`)"
            )
            raise HipLibraryUnavailable(_load_error)
        try:
            lib = ctypes.CDLL(str(LIB_PATH))
        except OSError as error:
            _load_error = f"cannot load {LIB_PATH}: {error}"
            raise HipLibraryUnavailable(_load_error) from error
        for name, (restype, argtypes) in SIGNATURES.items():
            fn = getattr(lib, name, None)
            if fn is None:
                _load_error = f"{LIB_PATH} lacks symbol {name}; rebuild it"
                raise HipLibraryUnavailable(_load_error)
            fn.restype = restype
            fn.argtypes = argtypes
        version = lib.pt_abi_version()
        if version != ABI_VERSION:
            _load_error = f"{LIB_PATH} has ABI version {version}, expected {ABI_VERSION}; rebuild it"
            raise HipLibraryUnavailable(_load_error)
        if sys.modules.get("torch") is not None:
            try:
                _bind_native(lib)
            except HipLibraryUnavailable as error:
                _load_error = str(error)
                raise
        _lib = lib
        return lib


def _bind_native(lib: ctypes.CDLL) -> None:
    """Loads the extension, once, and gives it the addresses of ``lib``'s entry points.  Called
    with the lock held."""

    global native, _native_tried
    if _native_tried:
        return
    try:
        found = importlib.import_module("picotron_amd._native")
        # the layout of torch's C++ objects is that of the version it was compiled against
        built, here = getattr(found, "TORCH_VERSION", None), str(sys.modules["torch"].__version__)
        if built is not None and built != here:
            raise ImportError(f"compiled against torch {built}, running under {here}")
    except ImportError as error:
        warnings.warn(f"the native launchers cannot be loaded ({error}); calls go through ctypes, with "
                      "more host time each (build them with `python -m picotron_amd.build`)",
                      RuntimeWarning, stacklevel=2)
        _native_tried = True
        return
    # bind() casts addresses to the prototypes of the header that the extension was compiled with
    version = getattr(found, "PT_ABI_VERSION", None)
    if version != ABI_VERSION:
        raise HipLibraryUnavailable(f"{found.__file__} has ABI version {version}, expected {ABI_VERSION}; rebuild it")
    for name in found.ENTRY_POINTS:
        found.bind(name, ctypes.cast(getattr(lib, name), c_void_p).value)
    native = found
    _launchers.update(
        pt_rmsnorm_fwd=native.rmsnorm_fwd,
        pt_rmsnorm_bwd=native.rmsnorm_bwd,
        pt_residual_rmsnorm_fwd=native.residual_rmsnorm_fwd,
        pt_residual_rmsnorm_bwd=native.residual_rmsnorm_bwd,
        pt_swiglu_fwd=native.swiglu_fwd,
        pt_swiglu_bwd=native.swiglu_bwd,
        pt_rope=native.rope,
        pt_cross_entropy=native.cross_entropy,
        pt_cross_entropy_shifted=native.cross_entropy,
        pt_cross_entropy_scale_grad=native.cross_entropy_scale_grad,
        pt_cross_entropy_shifted_scale_grad=native.cross_entropy_scale_grad,
    )
    _native_tried = True


def lib() -> ctypes.CDLL:
    """The loaded library; raises :class:`HipLibraryUnavailable` if it cannot be loaded."""

    return _lib if _lib is not None else _load()


def is_available() -> bool:
    try:
        lib()
    except HipLibraryUnavailable:
        return False
    return True


def unavailable_reason() -> str | None:
    if _lib is not None:
        return None
    try:
        lib()
    except HipLibraryUnavailable as error:
        return str(error)
    return None


def check(fn: str, rc: int) -> None:
    """Raise :class:`HipKernelError` with the library's message for a nonzero return."""

    if rc != PT_OK:
        message = lib().pt_last_error()
        raise HipKernelError(fn, rc, message.decode() if message else "")


_bound: dict[str, object] = {}


def raw_call(fn: str, *args) -> None:
    """Call entry point ``fn`` through ctypes and raise :class:`HipKernelError` on a nonzero
    return (the bound function object is looked up once per name)."""

    f = _bound.get(fn)
    if f is None:
        f = _bound[fn] = getattr(lib(), fn)
    rc = f(*args)
    if rc != PT_OK:
        check(fn, rc)


def extension():
    """The extension module, loading the library (or raising) and binding the extension when neither
    has happened yet; None when it cannot be loaded."""

    if not _native_tried:
        loaded = lib()
        with _lock:
            _bind_native(loaded)
    return native


def call(fn: str, *args):
    """One launch of entry point ``fn``: with raw arguments (integers, addresses) through ctypes;
    with tensors through its native launcher, which checks them, allocates the outputs and
    returns them -- or returns None when they are not the plain case that it takes or there is
    no launcher, and the caller goes its general route to :func:`raw_call`."""

    if not hasattr(args[0], "data_ptr"):
        return raw_call(fn, *args)
    launcher = _launchers.get(fn)
    if launcher is None:
        if extension() is None:
            return None
        launcher = _launchers[fn]
    out = launcher(*args)
    if type(out) is int:
        check(fn, out)
    return out
