"""The operators of kernels.py whose host side is native (csrc/host/native_ops.cpp -> lib/_tv_native.*.so), loaded at the first call on the GPU.

`ops.<name>(...)` returns the operator's result, or None where its operands are not the plain case: the caller then goes its own way."""
from __future__ import annotations

import importlib.machinery
import importlib.util

from . import _capi


class _Ops:
    def __getattr__(self, name):                 # (the first use alone: what is loaded lies in the instance)
        from .build import NATIVE, native_id
        _capi.lib()
        if not NATIVE.exists():
            raise _capi.TimeViperHipError(f"{NATIVE} is missing: run `python -m timeviper_amd.build`")
        loader = importlib.machinery.ExtensionFileLoader("_tv_native", str(NATIVE))
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_tv_native", loader))
        loader.exec_module(module)
        if getattr(module, "built_from", None) != native_id():
            raise _capi.TimeViperHipError(f"{NATIVE} was built from other sources or flags (tree {native_id()}): run `python -m timeviper_amd.build`")
        module.bind(str(_capi.lib_path()), _capi.TimeViperHipError)
        self.__dict__.update({k: v for k, v in vars(module).items() if not k.startswith("_")})
        if name not in self.__dict__:
            raise AttributeError(name)
        return self.__dict__[name]


ops = _Ops()
