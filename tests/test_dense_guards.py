"""When the native forms of float32 layers stand back: CPU checks of the conditions on the call."""
import contextlib
import importlib
from types import SimpleNamespace

import pytest
import torch
import torch.utils._device
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from pikv_amd import dense, ops


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


def test_compiled_call_is_noticed_without_a_graph_break():
    def f(x):
        return x + 1 if dense.ordinary_call() else x + 2

    assert torch.compile(f, backend="eager", fullgraph=True)(torch.zeros(())) == 2


@pytest.mark.parametrize("name", [
    "_C._len_torch_dispatch_stack", "_ops._len_torch_dispatch_stack_pre_dispatch", "_C._len_torch_function_stack",
    "_C._get_function_stack_at", "utils._device.DeviceContext", "nn.modules.module._has_any_global_hook",
    "_C._functorch.peek_interpreter_stack", "_C._has_storage", "autograd.forward_ad._current_level"])
def test_without_a_torch_internal_the_modules_run(monkeypatch, name):
    """A version of torch that lacks one of the internals: no error, and nothing counts as an ordinary call."""
    owner, attr = torch, name.split(".")
    for a in attr[:-1]:
        owner = getattr(owner, a)
    with monkeypatch.context() as m:
        m.delattr(owner, attr[-1])
        importlib.reload(dense)
        ordinary = dense.ordinary_call()
    importlib.reload(dense)
    assert ordinary is False and dense.ordinary_call()


def test_stream_without_the_raw_call(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: SimpleNamespace(cuda_stream=77))
    monkeypatch.setattr(ops, "_raw_stream", None, raising=False)
    assert ops._stream() == 77


@pytest.mark.parametrize("T,H,E,pays", [
    (1, 128, 4, True), (8192, 128, 16, True), (2048, 256, 64, True), (2048, 512, 64, True), (1024, 1024, 64, True),
    (128, 1536, 8, True), (128, 2048, 8, True),
    (8192, 128, 64, False), (65536, 128, 8, False), (8192, 512, 8, False), (2048, 1024, 64, False), (8192, 1024, 8, False),
    (256, 2048, 64, False), (1024, 2048, 4, False), (1, 4096, 4, False), (65536, 4096, 64, False)])
def test_router_rule_against_measured_sizes(T, H, E, pays):
    """Sizes where the native router was measured faster (pass and kernels) and where it was not."""
    assert dense.router_pays(T, H, E) is pays


@pytest.mark.parametrize("T,H,pays", [
    (1, 128, True), (8192, 128, True), (2048, 256, True), (1024, 512, True), (256, 1024, True), (128, 2048, True),
    (8192, 512, False), (2048, 1024, False), (512, 2048, False), (1, 4096, False), (8192, 4096, False)])
def test_key_projection_rule_against_measured_sizes(T, H, pays):
    assert dense.key_projection_pays(T, H) is pays


@pytest.mark.parametrize("T,H,N,pays", [
    (1, 256, 384, True), (64, 1024, 3072, True), (64, 2048, 6144, True), (32, 2560, 7680, True), (32, 3584, 5376, True),
    (16, 3072, 6144, True), (65, 256, 384, False), (64, 3072, 9216, False), (64, 4096, 6144, False), (32, 4096, 12288, False),
    (8, 8192, 12288, False), (1, 8192, 1024, False)])
def test_projection_rule_against_measured_sizes(T, H, N, pays):
    assert dense.projections_pay(T, H, N) is pays


@pytest.mark.parametrize("T,H,widths,pays", [
    (256, 512, (1024, 512, 512), True), (500, 1536, (2048, 1024, 1024), True), (4757, 256, (1536, 256, 256), True),
    (291, 1792, (2048, 1024, 1024), True), (1100, 2048, (768, 384, 384), True), (295, 3840, (2048, 512, 512), True),
    (307, 3584, (1024, 1024, 1024), True), (277, 4096, (2048, 512, 512), True), (397, 2048, (2048, 1024, 1024), True),
    (1280, 2048, (2048, 512, 512), True), (640, 3072, (4096, 1024, 1024), True), (1792, 2560, (1536, 384, 384), True),
    (896, 3840, (3584, 512, 512), True), (1000, 2048, (2048, 1024, 1024), True),
    (255, 512, (1024, 512, 512), False), (300, 3072, (2048, 768, 768), False), (330, 3072, (2048, 512, 512), False),
    (539, 3072, (1536, 256, 256), False), (639, 2304, (768, 768, 768), False), (261, 2048, (3584, 512, 512), False),
    (276, 4096, (1536, 256, 256), False), (266, 3072, (2048, 1024, 1024), False), (337, 3328, (1024, 1024, 1024), False),
    (871, 3072, (2048, 1024, 1024), False), (668, 3328, (3072, 1024, 1024), False), (1000, 3072, (1024, 1024, 1024), False),
    (4000, 3072, (1024, 1024, 1024), False)])
def test_tiled_rule_against_measured_sizes(T, H, widths, pays):
    """Sizes where one launch for q, k and v was measured no slower than three library calls, and where it was."""
    assert dense.tiled_pays(T, H, widths) is pays


@pytest.mark.parametrize("how", ["parameter", "buffer", "attribute"])
def test_frozen_weights_are_read_like_parameters(how):
    """Weights that were taken out of the parameters, as buffers or as plain attributes (data-parallel replicas hold theirs so)."""
    from pikv_amd.config import config
    from pikv_amd.moe import LoRALayer, PiKVMoE
    lin, lora = torch.nn.Linear(8, 4), LoRALayer(config["hidden_size"], config["hidden_size"], rank=2).eval()
    for m, names in ((lin, ("weight", "bias")), (lora, ("lora_A", "lora_B"))):
        for n in names if how != "parameter" else ():
            t = getattr(m, n).detach()
            delattr(m, n)
            m.register_buffer(n, t) if how == "buffer" else setattr(m, n, t)
    cpu = torch.device("cpu")
    assert dense.linear_ok(lin, 8, 4, cpu) and not dense.linear_ok(lin, 4, 8, cpu)
    assert PiKVMoE._lora_ok(None, lora, 2, cpu) and not PiKVMoE._lora_ok(None, lora, 4, cpu)
    lin.bias = None
    assert not dense.linear_ok(lin, 8, 4, cpu)


@pytest.mark.parametrize("T,H,E,tiled", [
    (33, 128, 4, True), (256, 128, 4, True), (128, 256, 4, True), (1025, 256, 4, True), (2048, 256, 8, True), (300, 384, 4, True),
    (5900, 384, 4, True), (1053, 512, 4, True), (2280, 512, 4, True), (520, 640, 4, True), (667, 1024, 4, True), (544, 1024, 6, True),
    (32, 128, 4, False), (257, 128, 4, False), (257, 256, 4, False), (1024, 256, 4, False), (511, 640, 4, False),     # another order
    (2049, 256, 4, False), (3000, 256, 4, False), (6145, 512, 2, False), (3073, 1024, 1, False), (8192, 384, 8, False),
    (743, 1536, 1, False), (633, 2048, 1, False), (716, 1536, 2, False), (548, 1280, 3, False), (1525, 1024, 1, False)])   # slower
def test_experts_rule_against_measured_sizes(T, H, E, tiled):
    """Sizes where the experts' products in one launch were measured faster and equal to the library's, and where not."""
    assert dense.experts_tiled(T, H, E) is tiled
