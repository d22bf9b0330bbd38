"""The native call path of the eager torch layer (``csrc/attnres_torch.cpp``).

``native.route`` / ``route_list`` / ``merge`` / ``block_step`` and the training
points' ``step`` / ``bwd_rows`` / ``bwd_defer`` / ``gather_seg`` launch one plain call and return its result, or return None with nothing done for any call that
is not plain (the caller then takes it through Python).  Loaded on first use;
without the built extension every function returns None, and the Python path
reports the missing library.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import threading
from pathlib import Path

PATH = Path(__file__).resolve().parent / "lib" / "_attnres_torch.so"
FUNCTIONS = ("route", "route_list", "merge", "block_step", "step", "bwd_rows", "bwd_defer", "gather_seg")

_lock = threading.Lock()


def _absent(*args):
    return None


class _Native:
    """The extension's functions as attributes, looked up once."""

    def __getattr__(self, name: str):
        if name not in FUNCTIONS:
            raise AttributeError(name)
        with _lock:
            mod = None
            if PATH.exists():
                loader = importlib.machinery.ExtensionFileLoader("_attnres_torch", str(PATH))
                mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("_attnres_torch", loader))
                loader.exec_module(mod)
            for fn in FUNCTIONS:
                self.__dict__[fn] = getattr(mod, fn) if mod is not None else _absent
        return self.__dict__[name]


native = _Native()
