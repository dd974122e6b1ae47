"""Where the float32 dense layers of the mixture-of-experts model take native kernels.

linear_group / adaptive_router / expert_combine (csrc/moe.hip) serve forward passes without autograd,
over modules that are what their class says: a subclass, a hook, an instance-level forward, autocast,
a functorch transform, forward-mode differentiation, a tracer or any other mode that watches torch's calls
all go through the module's own call.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.autograd import forward_ad
from torch.nn.modules import module as _module
from torch.utils._device import DeviceContext

MAX_LORA_RANK = 8
MAX_LAYERS = 20          # of one linear_group or expert_combine launch


def _no_hooks(m: nn.Module) -> bool:
    return not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                or "forward" in m.__dict__)


def plain(m, cls) -> bool:
    """m is exactly a `cls`, and calling it runs that class's forward and nothing else."""
    return type(m) is cls and _no_hooks(m)


def _watched() -> bool:
    """A function or dispatch mode (make_fx, a user's) sees torch's calls; to it the output of a kernel launched beside them is a
    constant.  A default device is a function mode too, but one that only places new tensors."""
    if torch._C._len_torch_dispatch_stack() or torch._ops._len_torch_dispatch_stack_pre_dispatch():
        return True
    n = torch._C._len_torch_function_stack()
    return n > 0 and any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(n))


def ordinary_call() -> bool:
    return not (_watched() or _module._has_any_global_hook() or torch.is_autocast_enabled("cuda") or torch.jit.is_tracing()
                or torch.compiler.is_compiling() or forward_ad._current_level >= 0
                or torch._C._functorch.peek_interpreter_stack() is not None)


def ordinary_tensor(t, device, dtype=torch.float32) -> bool:
    return (type(t) in (torch.Tensor, nn.Parameter) and t.device == device and t.dtype == dtype and t.is_contiguous()
            and torch._C._has_storage(t) and t.data_ptr() % 16 == 0)      # a batched tensor has none


def forward_only(x) -> bool:
    """A float32 GPU input of a pass that records nothing."""
    return not torch.is_grad_enabled() and x.is_cuda and ordinary_tensor(x, x.device) and ordinary_call()


def linear_ok(m, n_in: int, n_out: int, device) -> bool:
    """A plain nn.Linear of this shape with a bias, as linear_group reads it."""
    return (plain(m, nn.Linear) and m.bias is not None and m.weight.shape == (n_out, n_in)
            and ordinary_tensor(m.weight, device) and ordinary_tensor(m.bias, device))


def mlp_ok(seq, acts, sizes, device) -> bool:
    """A plain nn.Sequential of Linear layers of `sizes` with the activation classes `acts` behind them."""
    if not plain(seq, nn.Sequential):
        return False
    mods = list(seq)
    if len(mods) != len(sizes) - 1 + len(acts):
        return False
    for i in range(len(sizes) - 1):
        if not linear_ok(mods[2 * i], sizes[i], sizes[i + 1], device):
            return False
        if i < len(acts) and not plain(mods[2 * i + 1], acts[i]):
            return False
    return True
