"""The native host path (``csrc/host/cc1d_host.cpp``): loaded on the first call
with a GPU tensor and bound to the entry points of the library that ``_lib``
loaded. Its functions return ``NotImplemented`` for anything but the ordinary
case; the callers' Python code then runs as without it."""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
from pathlib import Path

from causal_conv1d_amd import _lib

_PATH = Path(__file__).resolve().parent / "_lib" / "cc1d_host.so"
_ENTRIES = ("cc1d_strerror", "cc1d_fwd", "cc1d_bwd_workspace_floats", "cc1d_bwd_typed", "cc1d_update",
            "cc1d_varlen_states")

_ext = None


def load():
    """The extension module (cached). Raises if it is missing, as the library does."""
    global _ext
    if _ext is None:
        if not _PATH.exists():
            raise RuntimeError(
                f"causal_conv1d_amd: native host path {_PATH} is not built; "
                "run `python causal-conv1d-mojo_amd/csrc/build.py`"
            )
        loader = importlib.machinery.ExtensionFileLoader("cc1d_host", str(_PATH))
        ext = importlib.util.module_from_spec(importlib.util.spec_from_loader("cc1d_host", loader))
        lib = _lib.load()
        ext.bind(*(ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _ENTRIES))
        _ext = ext
    return _ext


def native():
    return _ext if _ext is not None else load()
