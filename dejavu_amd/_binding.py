"""Loading of the in-tree kernel libraries with ctypes.  There is no fallback: a missing library raises."""
from __future__ import annotations

import ctypes
import os

import torch  # noqa: F401  (loads the HIP runtime that the libraries bind to)
from torch.utils._device import DeviceContext


def _watched() -> bool:
    """Whether a dispatch mode (make_fx, FlopCounterMode ..) or a function mode is active, which would see a library call and
    not a kernel's.  A default device is a function mode too, but one for the functions that make tensors."""
    return torch._C._len_torch_dispatch_stack() > 0 or any(
        type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(torch._C._len_torch_function_stack()))


def results_only(*tensors) -> bool:
    """Whether a kernel may stand in for a library call that also knows gradients, functional transforms, tracers,
    autocast, tensor subclasses and other devices: plain tensors of the current device, and none of these asked for."""
    here = torch.cuda.current_device() if torch.cuda.is_initialized() else -1
    grad = torch.is_grad_enabled()
    for t in tensors:
        if t is not None and (not t.is_cuda or t.device.index != here or (grad and t.requires_grad) or
                              type(t) not in (torch.Tensor, torch.nn.Parameter)):
            return False
    return (torch.autograd.forward_ad._current_level < 0 and torch._C._functorch.peek_interpreter_stack() is None and
            not torch.is_autocast_enabled() and not torch.jit.is_tracing() and not torch.compiler.is_compiling() and
            not _watched())


class DejavuHipError(RuntimeError):
    """An entry point of a kernel library returned a non-zero status."""


def load_library(path: str, signatures: dict) -> ctypes.CDLL:
    """signatures: name -> (restype, argtypes)."""
    if not os.path.exists(path):
        raise ImportError(f"{path} is missing: build it with `python -m dejavu_amd.build` "
                          "(there is no fallback implementation)")
    lib = ctypes.CDLL(path)
    for name, (restype, argtypes) in signatures.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    return lib
