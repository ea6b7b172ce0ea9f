"""Loading the compiled HIP libraries and calling their C entry points.

There is no fallback: if a library cannot be built or loaded, or a kernel launch
reports an error, an exception is raised.
"""
import ctypes
import os
from typing import Dict

import torch

from ..csrc import build as _build


class KernelError(RuntimeError):
    pass


_loaded: Dict[str, ctypes.CDLL] = {}


def library(name: str) -> ctypes.CDLL:
    """The shared library of module ``name``, built first if it is not there."""
    lib = _loaded.get(name)
    if lib is None:
        _build.ensure([name])
        path = _build.library_path(name)
        try:
            lib = ctypes.CDLL(path)
        except OSError as e:
            raise KernelError(f"cannot load the HIP library {path}: {e}") from None
        _loaded[name] = lib
    return lib


def loaded_libraries():
    return {n: _build.library_path(n) for n in _loaded}


# the two questions behind torch.cuda.current_stream(); looked up at the first launch, because a torch that was
# built without a GPU does not have them, and again in a forked process, which torch may refuse the device
_raw_stream = _current_device = None


def _forget_stream_functions():
    global _raw_stream, _current_device
    _raw_stream = _current_device = None


if hasattr(os, "register_at_fork"):
    os.register_at_fork(after_in_child=_forget_stream_functions)


def stream_handle() -> ctypes.c_void_p:
    """torch's current stream on its current device, asked anew at every launch.  As a number,
    not as a Stream object made for it: that object cost 4.5 us of an eager launch's 20
    (a prompt of 32 tokens and one token after it on a 12-layer model of 768 columns, 130
    launches: 2.58 ms of host time with it, 1.99 without)."""
    global _raw_stream, _current_device
    if _raw_stream is None:
        stream = torch.cuda.current_stream()   # starts the device, or says why it cannot (a forked process)
        if not hasattr(torch._C, "_cuda_getCurrentRawStream") or not hasattr(torch._C, "_cuda_getDevice"):
            return ctypes.c_void_p(stream.cuda_stream)
        _current_device, _raw_stream = torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream
    return ctypes.c_void_p(_raw_stream(_current_device()))


def ptr(t) -> ctypes.c_void_p:
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def check(code: int, what: str) -> None:
    if code != 0:
        raise KernelError(f"{what}: HIP error {code}")


def require_device(*tensors) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise KernelError("HIP kernels take device tensors only; there is no CPU path")


def require_contiguous(**tensors) -> None:
    for name, t in tensors.items():
        if t is not None and not t.is_contiguous():
            raise KernelError(f"{name} must be contiguous")
