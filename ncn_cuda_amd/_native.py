"""Loads _ncn_torch.so, the autograd nodes in native code (csrc/ncn_torch.cpp), and gives it the entry points of libncn_hip.so.

Its functions take the calls that need nothing done to their arguments and return None for every other one, which the
caller then runs through the Python node (same kernels, same results, same errors).
"""
import ctypes
import sys

from . import _lib

# in the order of `Library` in csrc/ncn_torch.cpp
ENTRIES = ("ncn_check_shape", "ncn_kernel_path_scalars", "ncn_error_string", "ncn_workspace_bytes",
           "ncn_workspace_bytes_stages", "ncn_forward", "ncn_backward", "ncn_forward_indexed", "ncn_backward_indexed",
           "ncn_stack_plan", "ncn_stack_forward", "ncn_stack_backward", "ncn_forward_radix", "ncn_backward_radix")


class _PythonNodes:
    """Stands in where _ncn_torch.so does not fit the torch beside it and cannot be built: takes no call."""

    @staticmethod
    def _none(*args):
        return None

    stage = table_stage = stack = radix = _none


_ext = None


def ext():
    """The extension module, loaded and bound once; built first if it is missing or made from other sources.  Where that cannot
    be done the nodes in Python run instead, which is said once and remembered: the same kernels, more host time."""
    global _ext
    if _ext is None:
        lib = _lib.load()   # the kernels themselves have no substitute: this raises
        try:
            _ext = _load(lib)
        except Exception as exc:
            print(f"ncn_cuda_amd: warning: autograd nodes run in Python, _ncn_torch.so cannot be used: {exc}", file=sys.stderr)
            _ext = _PythonNodes
    return _ext


def _load(lib):
    from . import _build
    if not _build.have_sources():
        made_for = _build.torch_library_for()
        if made_for != _build.torch_in_use():
            raise ImportError("it is missing" if made_for is None else f"it was built for torch and Python {made_for}")
    elif _build.torch_library_id() != _build.torch_source_id():
        if _build.have_cxx():
            print("ncn_cuda_amd: building _ncn_torch.so with g++ (half a minute)", file=sys.stderr)
        _build.build_torch(force=False)
    from . import _ncn_torch
    _ncn_torch.bind(tuple(ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in ENTRIES))
    return _ncn_torch
