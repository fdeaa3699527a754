"""The native dispatch module (csrc/host/snnf_dispatch.cpp -> lib/_snnf_dispatch.so): operator calls and internal-layout calls
whose signature has been seen run from C++; everything else runs the Python implementations, which this module hands it.

The module is an accelerator of the host side and nothing more: without it (not built, or built against another PyTorch) every call
runs its Python implementation on the same kernels of libsnnf.so."""
from __future__ import annotations

import importlib
import importlib.machinery
import importlib.util
import warnings
from typing import Callable, Optional

from . import _lib

DISPATCH_PATH = _lib.PKG_DIR / "lib" / "_snnf_dispatch.so"


class _Absent:
    """Stands in for the extension where there is none: it knows no call."""

    def __getattr__(self, name: str) -> Callable:
        if name.startswith("__"):
            raise AttributeError(name)
        return lambda *args: None


_MODULE = None


def available() -> bool:
    return _lib.library_available() and DISPATCH_PATH.exists()


def load():
    """The extension, or None where there is none or it cannot be loaded (which is said once). Loading it registers the operators'
    GPU implementations."""
    global _MODULE
    if _MODULE is None:
        _MODULE = _Absent()
        if available():
            try:
                _lib.lib()
                loader = importlib.machinery.ExtensionFileLoader("_snnf_dispatch", str(DISPATCH_PATH))
                spec = importlib.util.spec_from_file_location("_snnf_dispatch", str(DISPATCH_PATH), loader=loader)
                loaded_module = importlib.util.module_from_spec(spec)
                loader.exec_module(loaded_module)
                _MODULE = loaded_module
            except (ImportError, OSError) as exc:
                warnings.warn(f"{DISPATCH_PATH} cannot be loaded, calls run their Python implementations (build it again with "
                              f"`python triton-snn-fusion_amd/build.py`): {exc}", RuntimeWarning, stacklevel=2)
    return loaded()


def module():
    """What internal-layout calls are handed to: the extension, connected, or its stand-in."""
    if _MODULE is None and load() is not None:
        # The operator layer connects the extension (`connect` below) when it is imported: whoever loads the extension imports it.
        importlib.import_module(".runtime.snn_custom_ops", __package__)
    return _MODULE


def loaded():
    """The extension if something has loaded it, else None."""
    return None if isinstance(_MODULE, _Absent) else _MODULE


def connect(slow: Callable, pack: Callable, plane: Callable, workspace: Callable) -> Optional[object]:
    """Hands the Python implementations to the extension: operator calls, weight packing, plane matrices, workspaces."""
    m = load()
    if m is not None:
        m.connect(slow, pack, plane, workspace)
    return m
