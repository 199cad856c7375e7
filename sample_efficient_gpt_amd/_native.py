"""Loader of ``_segpt_torch.so``, the native host side of the op for PyTorch callers (csrc/torch_binding.cpp): argument
checks, allocation, launch and autograd node.  Like the kernel library there is no fallback: if it was not built,
loading raises."""

from __future__ import annotations

import importlib.util
import os
import threading

from . import _lib

MODULE_PATH = os.path.join(_lib.PKG_DIR, "_segpt_torch.so")

_module = None
_lock = threading.Lock()


def load():
    """Load (once) and return the native module; raises if it was not built."""
    global _module
    if _module is not None:
        return _module
    with _lock:
        if _module is not None:
            return _module
        _lib.load()
        if not os.path.exists(MODULE_PATH):
            raise RuntimeError(f"{MODULE_PATH} not found: build it with `python -m sample_efficient_gpt_amd.build`. There is no fallback path.")
        import torch  # noqa: F401  (its libraries have to be in the process first)

        spec = importlib.util.spec_from_file_location("_segpt_torch", MODULE_PATH)
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        mod.set_error_class(_lib.SegptError)
        _module = mod
    return _module
