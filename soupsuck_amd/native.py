"""The native autograd nodes (``_native.so``, csrc/torch/nodes.cpp), loaded on first use.

They run the layers' forward and backward without the interpreter; the Python nodes they
stand for remain for timing hooks (``_lib.hooks``) and special variants.  A missing
extension is an error, as a missing kernel library is.
"""

from . import _lib

_module = None


def nodes():
    """The extension module, or None while timing hooks want the Python nodes' calls."""
    global _module
    if _lib.hooks:
        return None
    if _module is None:
        _lib.load()
        try:
            from . import _native
        except ImportError as exc:
            raise RuntimeError("soupsuck_amd: the native nodes are not built; run "
                               "`python -m soupsuck_amd.build` first") from exc
        _module = _native
    return _module
