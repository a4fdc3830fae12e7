"""The operators of kernels.py whose host side is native (csrc/host/native_ops.cpp -> lib/_tv_native.*.so), loaded at the first call on the GPU.

`ops.<name>(...)` returns the operator's result, or None where its operands are not the plain case: the caller then goes its own way, through ctypes to the same
entries.  Where the extension is missing, was built from other sources or cannot be loaded (it needs a C++ compiler, Python.h and torch's headers, which the library does
not), that holds for every call, and a warning says so once."""
from __future__ import annotations

import importlib.machinery
import importlib.util
import warnings

from . import _capi


def _load():
    from .build import NATIVE, native_id
    if not NATIVE.exists():
        raise ImportError("it is not built")
    loader = importlib.machinery.ExtensionFileLoader("_tv_native", str(NATIVE))
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_tv_native", loader))
    loader.exec_module(module)
    if getattr(module, "built_from", None) != native_id():
        raise ImportError(f"it was built from other sources or flags (tree {native_id()})")
    module.bind(str(_capi.lib_path()), _capi.TimeViperHipError)
    return module


class _Ops:
    def __getattr__(self, name):                 # (the first use alone: what is loaded lies in the instance)
        if name.startswith("__"):
            raise AttributeError(name)
        _capi.lib()
        if "native" not in self.__dict__:
            try:
                self.native = _load()
            except (ImportError, OSError, RuntimeError) as e:
                self.native = None
                warnings.warn(f"timeviper_amd: the native host side of the operators is not used, calls go through ctypes: {e}; `python -m timeviper_amd.build` makes it",
                              RuntimeWarning, stacklevel=2)
        self.__dict__[name] = getattr(self.native, name) if self.native else lambda *a: None
        return self.__dict__[name]


ops = _Ops()
