"""The native host path of the ops (bpt_amd/csrc/bptop.cpp -> bptop.so): a call whose plan is known is checked, allocated and
launched there, and its backward runs on autograd's thread without the interpreter.  What it may launch is what
bpt_amd/graphop.py chose and left in its table; see there.  There is no fallback: without the built module the import fails.
"""
import importlib.machinery
import importlib.util
import os

import torch  # noqa: F401  (the module links against its libraries)

from ._build import OP_SO


def _load():
    if not os.path.exists(OP_SO):
        raise ImportError(f"bptop is not built ({OP_SO} missing): run `python -m bpt_amd._build`")
    loader = importlib.machinery.ExtensionFileLoader("bptop", OP_SO)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("bptop", OP_SO, loader=loader))
    loader.exec_module(module)
    return module


native = _load()
