"""Native eager dispatch of the custom ops (csrc/sihc_torch.cpp).

`native(op, name)` keeps `op` the registered `sihc::` custom op it is, with its schema, fake
and autograd rules, and gives its Python call a short cut: where every argument is a plain
packed GPU tensor of an accepted shape and no tracing, dispatch or function mode, functorch
transform or forward-mode tangent is in force, a C++ autograd node launches the kernels
directly; any other call, and every call with keyword arguments, runs the op as before. So does
every call of an op that the program gave a kernel, an autograd rule or an autocast rule of its
own. One
training pass of event_write_read at batch 8 x 768 channels took 123 us of host time through the
Python op and its kernels 40 us.
"""
from __future__ import annotations

import importlib.util
from pathlib import Path
from typing import Callable, Optional

from torch.compiler import is_compiling
from torch.library import CustomOpDef

from ._lib import lib

NATIVE_PATH = Path(__file__).resolve().with_name("_sihc_torch.so")
_module = None


def module():
    """The extension, loaded once. Raises if it is absent: there is no silent slow path."""
    global _module
    if _module is None:
        if not NATIVE_PATH.exists():
            raise RuntimeError(f"{NATIVE_PATH} is missing: build it with "
                               "`python residual-stream-burden_amd/build.py`")
        lib()  # the library that the extension calls, its version checked
        spec = importlib.util.spec_from_file_location("_sihc_torch", NATIVE_PATH)
        loaded = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(loaded)
        _module = loaded
    return _module


def _declined(*args):
    return NotImplemented


class _NativeOp(CustomOpDef):
    """A custom op whose plain eager calls take the native entry."""

    # What replaces the op's own kernel or rule ends the short cut. (A kernel or autocast rule
    # under a GPU dispatch key is seen by the entry itself, however it was registered.)
    def register_kernel(self, device_types, fn=None, /):
        if device_types is None:
            self._sihc_entry = _declined
        return super().register_kernel(device_types, fn)

    def register_autograd(self, backward, /, **kwargs):
        self._sihc_entry = _declined
        return super().register_autograd(backward, **kwargs)

    def __call__(self, *args, **kwargs):
        if not kwargs and not is_compiling():
            entry = self._sihc_entry
            if entry is None:
                entry = self._sihc_entry = self._sihc_load()
            out = entry(*args)
            if out is not NotImplemented:
                return out
        return super().__call__(*args, **kwargs)


def native(op: CustomOpDef, name: str, adapt: Optional[Callable] = None) -> CustomOpDef:
    """Give `op` the native entry `name`; `adapt(entry)` may wrap it (more checks, more
    arguments) in a function that returns NotImplemented where it does not apply."""
    def load():
        entry = module().entry(name, op._qualname)
        return entry if adapt is None else adapt(entry)

    op.__class__ = _NativeOp
    op._sihc_entry, op._sihc_load = None, load
    return op
