"""The operators' native host path (``_fla_torch.so``, csrc/fla_torch.cc).

``product``, ``mapped`` and ``polynomial`` run an operator -- tests, allocation, the call into ``libfla_gfx950.so`` and,
when a gradient is wanted, the autograd node -- and return its output, or None for a call that is not the
plain case (the caller then runs the Function's Python forward, which also raises what there is to
raise).  The extension is loaded at the first call with a tensor on the GPU; a missing one raises.
"""

from __future__ import annotations

import importlib.util
import os

from . import _lib

_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_fla_torch.so")
_module = None


def _load():
    global _module
    with _lib._lock:
        if _module is None:
            if not os.path.exists(_PATH):
                raise RuntimeError(f"{_PATH} is missing: build it with `python -m flashy_linear_attention_amd.build`")
            spec = importlib.util.spec_from_file_location("flashy_linear_attention_amd._fla_torch", _PATH)
            module = importlib.util.module_from_spec(spec)
            spec.loader.exec_module(module)
            _module = module
    return _module


def entry(name: str):
    """The extension's function `name`, behind a stub that loads the extension and then steps aside: callers read
    ``_native.<name>`` at each call."""

    def stub(*args):
        if not any(getattr(a, "is_cuda", False) for a in args):
            return None
        _lib.load()  # (checks the library's ABI)
        module = _load()
        globals()[name] = getattr(module, name)
        return globals()[name](*args)

    return stub


product = entry("product")
mapped = entry("mapped")
polynomial = entry("polynomial")
