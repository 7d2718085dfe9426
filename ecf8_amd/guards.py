"""When a call may leave torch's dispatcher for a HIP kernel: the checks
shared by the wrappers that replace torch operations and fall back to them."""

from __future__ import annotations

import torch
from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _function_modes() -> bool:
    return bool(torch._C._len_torch_function_stack()) and not all(
        type(m) is DeviceContext for m in _get_current_function_mode_stack())


def untracked() -> bool:
    """No tracer, dispatch or function mode (but a default device), dual level
    or autocast region is active."""
    return not (torch._C._len_torch_dispatch_stack() or forward_ad._current_level >= 0
                or _function_modes() or torch.is_autocast_enabled("cuda") or torch.jit.is_tracing()
                or torch.compiler.is_compiling())


def takes(tensors, dtype=torch.bfloat16, grad=False) -> bool:
    """Plain, non-empty, 16-byte aligned CUDA tensors of one dtype on one
    device that functorch does not wrap and (unless ``grad``) autograd does
    not follow."""
    dev, followed = tensors[0].device, torch.is_grad_enabled() and not grad
    return all(type(t) in _PLAIN and t.is_cuda and t.device == dev and t.dtype == dtype
               and t.numel() > 0 and not (followed and t.requires_grad)
               and not torch._C._functorch.is_functorch_wrapped_tensor(t)
               and t.data_ptr() % 16 == 0 for t in tensors)


def bare(mod, cls) -> bool:
    """``mod`` is exactly a ``cls`` without hooks or a forward of its own, so
    its forward may be computed without calling it."""
    return (type(mod) is cls and "forward" not in mod.__dict__
            and not torch.nn.modules.module._has_any_global_hook()
            and not (mod._forward_hooks or mod._forward_pre_hooks or mod._backward_hooks
                     or mod._backward_pre_hooks))
