"""The native host path (``ebr_amd/csrc/ebr_host.cpp``, built to ``ebr_amd/_lib/ebr_host.so``): autograd nodes and
launches of the GPU ops without Python in between.

``module()`` is the loaded extension, or None when it is not there or does not load with this torch: the Python layer
then runs the same kernels of ``libebr_attn.so`` (and raises if that is missing). Each of its functions returns None for
a call that the Python layer has to take (see the source's header); callers go on in Python then.

``GRADS``: the Python formulas of the native nodes' gradients, by node. A native node whose backward runs under a
transform (``is_grads_batched``), a mode or a hook, or with cotangents that are no plain tensors, calls its formula: the
saved values, then the cotangents (None where there is none), and gets the inputs' gradients.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import threading
import warnings
from typing import Callable, Dict

import torch  # noqa: F401  (the extension links against torch's libraries)

from ebr_amd import _capi

NAME = "ebr_host"
PATH = _capi.LIB_PATH.with_name(NAME + ".so")

GRADS: Dict[str, Callable] = {}


def gradient(node: str) -> Callable[[Callable], Callable]:
    """Registers the decorated function as a native node's Python gradient."""

    def register(fn: Callable) -> Callable:
        GRADS[node] = fn
        return fn

    return register


_LOCK = threading.Lock()
_TRIED = False
_MODULE = None


def _load():
    global _TRIED, _MODULE
    with _LOCK:
        if _TRIED:
            return _MODULE
        try:
            _capi.load()  # the extension calls the library's entry points
            loader = importlib.machinery.ExtensionFileLoader(NAME, str(PATH))
            spec = importlib.util.spec_from_file_location(NAME, str(PATH), loader=loader)
            mod = importlib.util.module_from_spec(spec)
            loader.exec_module(mod)
            _MODULE = mod
        except (ImportError, OSError, RuntimeError) as exc:
            if PATH.exists():
                warnings.warn(f"ebr_amd: {PATH} does not load ({exc}); the slower Python host path runs instead "
                              "(rebuild with `python -m ebr_amd.build`)", RuntimeWarning, stacklevel=3)
        _TRIED = True
        return _MODULE


def module():
    return _MODULE if _TRIED else _load()


__all__ = ["GRADS", "gradient", "module"]
