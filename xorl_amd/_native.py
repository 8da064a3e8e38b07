"""The compiled host path (csrc/xq_torch.cpp) as a Python module.

Its functions take a module of this package and tensors, run the forward through the library and record the backward as a
C++ autograd node; they return None for calls that they leave to the Python path.  Like the kernel library it has no
fallback: if it has not been built, the first call raises.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import inspect
import os

from . import _C


PATH = os.path.join(os.path.dirname(_C.LIB_PATH), "xq_torch.so")

_module = None


def program(cls, *names):
    """A module class and the methods whose work the native path does without calling them, as the class defines them.  A module
    on which one of them is another (a subclass, an instance attribute, a patched class) is left to the Python path."""
    return cls, tuple((n, inspect.getattr_static(cls, n)) for n in names)


def _load():
    global _module
    _C.lib()
    if not os.path.exists(PATH):
        raise RuntimeError(f"{PATH} is missing: build it with `python -m xorl_amd.csrc.build`")
    from . import functional
    from .qlora import linear, moe_experts

    loader = importlib.machinery.ExtensionFileLoader("xq_torch", PATH)
    m = importlib.util.module_from_spec(importlib.util.spec_from_file_location("xq_torch", PATH, loader=loader))
    loader.exec_module(m)
    m.init(_C.XqError, functional.__dict__, linear.NATIVE_PROGRAMS, moe_experts.NATIVE_PROGRAMS)
    _module = m
    return m


def native():
    return _module or _load()
