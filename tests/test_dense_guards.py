"""When the native forms of float32 layers stand back: CPU checks of the conditions on the call."""
import contextlib

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from pikv_amd import dense


class _FunctionMode(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _DispatchMode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("mode,ordinary", [
    (contextlib.nullcontext, True), (torch.no_grad, True), (torch.inference_mode, True),
    (lambda: torch.device("cpu"), True),                    # a default device is a function mode that runs nothing else
    (_FunctionMode, False), (_DispatchMode, False), (torch._subclasses.FakeTensorMode, False),
], ids=["plain", "no_grad", "inference", "device", "function", "dispatch", "fake"])
def test_ordinary_call_under_modes(mode, ordinary):
    with mode():
        assert dense.ordinary_call() is ordinary
    assert dense.ordinary_call()


@pytest.mark.parametrize("tracing", ["real", "fake", "symbolic"])
@pytest.mark.parametrize("pre_dispatch", [False, True])
def test_make_fx_is_noticed(tracing, pre_dispatch):
    """A traced call takes torch operations: what a native kernel returns would be a constant of the graph."""
    from torch.fx.experimental.proxy_tensor import make_fx
    seen = []

    def f(x):
        seen.append(dense.ordinary_call())
        return x + 1

    make_fx(f, tracing_mode=tracing, pre_dispatch=pre_dispatch)(torch.ones(3))
    assert seen and not any(seen)
