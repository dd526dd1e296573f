"""Loads the C++ operator library (libgs.so) into torch.  There is no fallback:
a missing library is an import error that says how to build it."""
import importlib.util
import os

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
SO_PATH = os.path.join(_HERE, "lib", "libgs.so")
PYTHON_PATH = os.path.join(_HERE, "lib", "_gs_python.so")
_loaded = False
native = None      # the module _gs_python


def load() -> None:
    global _loaded, native
    if _loaded:
        return
    missing = [p for p in (SO_PATH, PYTHON_PATH) if not os.path.exists(p)]
    if missing:
        raise ImportError(
            f"{missing[0]} is missing: build it with `python -c 'import __graft_entry__ as g; "
            "g.build()'` (make -C gsampler_amd/csrc && python gsampler_amd/csrc/host/build.py)")
    torch.classes.load_library(SO_PATH)
    spec = importlib.util.spec_from_file_location("_gs_python", PYTHON_PATH)
    native = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(native)
    _loaded = True
