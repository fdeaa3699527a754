"""The native dispatch module (csrc/host/snnf_dispatch.cpp -> lib/_snnf_dispatch.so): operator calls and internal-layout calls
whose signature has been seen run from C++; everything else runs the Python implementations, which this module hands it."""
from __future__ import annotations

import importlib
import importlib.machinery
import importlib.util
from typing import Callable, Optional

from . import _lib

DISPATCH_PATH = _lib.PKG_DIR / "lib" / "_snnf_dispatch.so"

_MODULE = None


def available() -> bool:
    return _lib.library_available()


def module():
    """The loaded extension; raises when it has not been built. Loading it registers the operators' GPU implementations."""
    global _MODULE
    if _MODULE is None:
        if not available():
            raise RuntimeError(f"{DISPATCH_PATH} not found; build it with `python triton-snn-fusion_amd/build.py`")
        _lib.lib()
        loader = importlib.machinery.ExtensionFileLoader("_snnf_dispatch", str(DISPATCH_PATH))
        spec = importlib.util.spec_from_file_location("_snnf_dispatch", str(DISPATCH_PATH), loader=loader)
        loaded = importlib.util.module_from_spec(spec)
        loader.exec_module(loaded)
        _MODULE = loaded
        # The operator layer connects the extension (`connect` below) when it is imported: whoever loads the extension imports it.
        importlib.import_module(".runtime.snn_custom_ops", __package__)
    return _MODULE


def loaded():
    """The extension if something has loaded it, else None."""
    return _MODULE


def connect(slow: Callable, pack: Callable, plane: Callable, workspace: Callable) -> Optional[object]:
    """Hands the Python implementations to the extension: operator calls, weight packing, plane matrices, workspaces."""
    m = module()
    m.connect(slow, pack, plane, workspace)
    return m
