"""The native front of the operators (``csrc/hstu_native.cpp``), loaded on first use.

``native.front`` is the extension module.  Its functions serve the usual call of an operator and return ``None`` for any
other, which the operators of this package then handle in Python.
"""

import importlib.machinery
import importlib.util
import os

from ..build import LIB_PATH, LINEAR_LIB_PATH, NATIVE_PATH


class _Unloaded:
    """Stands in until the first function is asked for, so that the package imports before it is built."""

    def __getattr__(self, name):
        global front
        for path in (NATIVE_PATH, LIB_PATH, LINEAR_LIB_PATH):
            if not os.path.exists(path):
                raise RuntimeError(f"{path} is missing: build it with __graft_entry__.build().  There is no fallback.")
        loader = importlib.machinery.ExtensionFileLoader("hstu_native", NATIVE_PATH)
        module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("hstu_native", NATIVE_PATH, loader=loader))
        loader.exec_module(module)
        front = module
        return getattr(module, name)


front = _Unloaded()
