"""The native call path of the eager torch layer (``csrc/attnres_torch.cpp``).

``native.route`` / ``route_list`` / ``merge`` / ``block_step`` and the training
points' ``step`` / ``bwd_rows`` / ``bwd_defer`` / ``gather_seg`` launch one
plain call and return its result, or return None with nothing done for any
call that is not plain (the caller then takes it through Python).  Loaded on
first use.  Without the built extension every function returns None and the
calls take the ctypes path, which reports a missing library; so they do, with
a warning, where the extension does not load or was built for another torch.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import threading
import warnings
from pathlib import Path

# named for this interpreter: one built for another Python is not found
NAME = "_attnres_torch" + importlib.machinery.EXTENSION_SUFFIXES[0]
PATH = Path(__file__).resolve().parent / "lib" / NAME
FUNCTIONS = ("route", "route_list", "merge", "block_step", "step", "bwd_rows", "bwd_defer", "gather_seg")

_lock = threading.Lock()


def _absent(*args):
    return None


def _load(path: Path):
    """The extension module, or None where it is absent or not of this torch (with a warning)."""
    if not path.exists():
        return None
    import torch

    try:
        loader = importlib.machinery.ExtensionFileLoader("_attnres_torch", str(path))
        mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("_attnres_torch", loader))
        loader.exec_module(mod)
        if mod.torch_version != torch.__version__:
            raise ImportError(f"built for torch {mod.torch_version}, this is {torch.__version__}")
    except ImportError as e:
        warnings.warn(f"{path}: the native call path is off, eager calls take the slower ctypes path: {e} "
                      "(python -m kotodama_amd.build builds it again)", RuntimeWarning, stacklevel=3)
        return None
    return mod


class _Native:
    """The extension's functions as attributes, looked up once."""

    def __getattr__(self, name: str):
        if name not in FUNCTIONS:
            raise AttributeError(name)
        with _lock:
            if name not in self.__dict__:  # another thread may have been first
                mod = _load(PATH)
                self.__dict__.update({fn: getattr(mod, fn, _absent) for fn in FUNCTIONS})
        return self.__dict__[name]


native = _Native()
