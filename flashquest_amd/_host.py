"""The operators' native host path (csrc/host_torch.cpp).

One C++ call builds the descriptors, allocates the outputs and calls the HIP
library, in place of the ctypes path's per-tensor Python.  It answers None for
everything outside its plain case, and the operators then take the ctypes path;
without the module (not built, or built for another torch, interpreter or library)
they always do.  Either way the same entries of the same library run.
"""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os
import warnings

from . import _lib as L

_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_lib", "_fq_host.so")
_module = None
_loaded = False


def _load():
    """The module bound to the loaded library."""
    loader = importlib.machinery.ExtensionFileLoader("_fq_host", _PATH)
    m = importlib.util.module_from_spec(importlib.util.spec_from_loader("_fq_host", loader))
    loader.exec_module(m)
    lib = L.lib()
    m.bind({name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in L.SIGNATURES})
    return m


def module():
    """The native module bound to the loaded library, or None when it is not built
    or does not load here (said once)."""
    global _module, _loaded
    if not _loaded:
        if os.path.exists(_PATH):
            try:
                _module = _load()
            except (ImportError, KeyError, ValueError) as e:      # another torch or interpreter, another library
                warnings.warn(f"the native host path is not used, build it again: {e!r}", RuntimeWarning, stacklevel=2)
        _loaded = True
    return _module
