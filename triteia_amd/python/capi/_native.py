"""Loader of the native op binding (triteia_amd/csrc/torch_ops.cpp), built in-tree next to libtriteia_hip.so."""
import importlib.machinery
import importlib.util
import os

from . import _ffi

LIB_PATH = os.path.join(os.path.dirname(_ffi.LIB_PATH), "triteia_torch.so")
_module = None


def native():
    """The loaded module; raises RuntimeError if it has not been built.  Its functions return None for what they leave
    to the Python path of the op that calls them."""
    global _module
    if _module is None:
        _ffi.lib()
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(f"{LIB_PATH} not found: build it with `python -m triteia_amd.build`")
        loader = importlib.machinery.ExtensionFileLoader("triteia_torch", LIB_PATH)
        spec = importlib.util.spec_from_file_location("triteia_torch", LIB_PATH, loader=loader)
        module = importlib.util.module_from_spec(spec)
        loader.exec_module(module)
        _module = module
    return _module
