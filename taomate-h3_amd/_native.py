"""Loader of the native tensor wrappers (csrc/torch_ops.cpp, built in-tree by
build.py next to the kernel library it calls).  There is no fallback: a GPU call
without the built module raises, as a call without the kernel library does."""

from __future__ import annotations

import importlib.machinery
import importlib.util
import threading
from pathlib import Path
from types import ModuleType

from . import _lib

NAME = "_h3q_torch"
PATH = Path(__file__).resolve().parent / f"{NAME}.so"

_lock = threading.Lock()
_module: ModuleType | None = None


def module() -> ModuleType:
    global _module
    if _module is None:
        with _lock:
            if _module is None:
                _lib.lib()  # the kernel library first: its own error if it is missing
                if not PATH.exists():
                    raise RuntimeError(f"{PATH.name} is not built: run `python taomate-h3_amd/build.py`")
                loader = importlib.machinery.ExtensionFileLoader(NAME, str(PATH))
                spec = importlib.util.spec_from_file_location(NAME, str(PATH), loader=loader)
                native = importlib.util.module_from_spec(spec)
                loader.exec_module(native)
                _module = native
    return _module
