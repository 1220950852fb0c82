"""The host side of the hot operators as a compiled extension (``csrc/torch_host.cpp``): argument checks, allocation, launches
through libfla_hip.so and the autograd nodes.  Built in-tree by ``flash-linear-attention_amd/build.py`` beside libfla_hip.so;
there is no fallback.  Every function returns ``None`` where a call needs a conversion first."""
import importlib.machinery
import importlib.util
import os

import torch  # noqa: F401  (loads the libraries the extension links against)

from . import _backend as be

_PATH = os.path.join(os.path.dirname(be.lib_path()), "_fla_host.so")
_mod = None


def host():
    """The loaded extension; raises if it has not been built."""
    global _mod
    if _mod is None:
        be.lib()
        if not os.path.exists(_PATH):
            raise RuntimeError(f"fla_amd: host extension not built ({_PATH} is missing). "
                               "Run `python flash-linear-attention_amd/build.py` (needs hipcc); there is no CPU fallback.")
        loader = importlib.machinery.ExtensionFileLoader("_fla_host", _PATH)
        mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("_fla_host", loader))
        loader.exec_module(mod)
        if mod.ABI_VERSION != be.ABI_VERSION:
            raise RuntimeError("fla_amd: _fla_host.so ABI version mismatch; rebuild it")
        _mod = mod
    return _mod
