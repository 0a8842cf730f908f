"""Loader of the native host path, ``_fox_torch`` (csrc/fox_torch.cpp): the operators' entry points with allocation, launches
and autograd nodes in C++.  Loaded lazily and exactly once; like the kernel library it has no substitute: a missing file
raises ``RuntimeError``.
"""
from __future__ import annotations

import importlib.machinery
import importlib.util
import threading

import torch  # noqa: F401  (the extension links against torch's libraries, which this import brings in)

from ._lib import LIB_PATH

EXT_PATH = LIB_PATH.with_name("_fox_torch.so")

_ext = None
_bounds = None   # the list of an active record_pruning_bounds()
_lock = threading.Lock()


def load():
    """The extension module."""
    global _ext
    if _ext is not None:
        return _ext
    with _lock:
        if _ext is None:
            if not EXT_PATH.exists():
                raise RuntimeError(f"{EXT_PATH} is missing: build it with `python forgetting-transformer_amd/build.py` "
                                   "(there is no fallback implementation)")
            loader = importlib.machinery.ExtensionFileLoader("_fox_torch", str(EXT_PATH))
            spec = importlib.util.spec_from_loader("_fox_torch", loader)
            module = importlib.util.module_from_spec(spec)
            loader.exec_module(module)
            module.record_bounds(_bounds)
            _ext = module
    return _ext


def record_bounds(records) -> None:
    """Have the native nodes' backwards add their pruning bounds to ``records`` (None: to nothing)."""
    global _bounds
    with _lock:
        _bounds = records
        if _ext is not None:
            _ext.record_bounds(records)
