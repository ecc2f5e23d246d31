"""The C++ side of the operators: `_torch_ops.so` (csrc/torch/*.cpp), torch operators and autograd nodes over the C ABI.

Loaded when this module is imported if it has been built; `native()` returns it or raises as `_lib.lib()` does.
"""
from __future__ import annotations

from pathlib import Path

import torch  # noqa: F401  (its libraries must be loaded before the extension that links against them)

from . import _lib

EXT_PATH = Path(__file__).resolve().parent / "_torch_ops.so"
_MODULE = None

if EXT_PATH.exists() and _lib.LIB_PATH.exists():
    from . import _torch_ops as _MODULE  # type: ignore[no-redef]


def native():
    if _MODULE is None:
        _lib.lib()  # names the missing library, if it is that one
        raise _lib.MaltosHipError(f"{EXT_PATH} is missing: build it with `python -m maltos_amd.build`. "
                                  "maltos_amd has no CPU or eager fallback.")
    return _MODULE
