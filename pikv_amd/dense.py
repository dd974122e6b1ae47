"""Where the float32 dense layers of the mixture-of-experts model take native kernels.

linear_group / adaptive_router / expert_combine (csrc/moe.hip) serve forward passes without autograd,
over modules that are what their class says: a subclass, a hook, an instance-level forward, autocast,
a functorch transform, forward-mode differentiation, a tracer or any other mode that watches torch's calls
all go through the module's own call.
"""
from __future__ import annotations

from functools import lru_cache, reduce

import torch
import torch.nn as nn
from torch.autograd import forward_ad

from . import ops

try:
    from torch.utils._device import DeviceContext as _DeviceContext
except ImportError:
    _DeviceContext = None


def _internal(path: str):
    """torch.<path>, or None in a version of torch that does not have it."""
    return reduce(lambda o, name: getattr(o, name, None), path.split("."), torch)


# What tells whether something watches a call is internal to torch.  Where a name is missing the answer is yes:
# every layer takes its module's own call.
_dispatch_modes = _internal("_C._len_torch_dispatch_stack")
_pre_dispatch_modes = _internal("_ops._len_torch_dispatch_stack_pre_dispatch")
_function_modes = _internal("_C._len_torch_function_stack")
_function_mode_at = _internal("_C._get_function_stack_at")
_has_global_hook = _internal("nn.modules.module._has_any_global_hook")
_transforms = _internal("_C._functorch.peek_interpreter_stack")
_has_storage = _internal("_C._has_storage")
_is_compiling, _is_tracing, _is_autocast = torch.compiler.is_compiling, torch.jit.is_tracing, torch.is_autocast_enabled
_KNOWN = (hasattr(forward_ad, "_current_level")
          and None not in (_dispatch_modes, _pre_dispatch_modes, _function_modes, _function_mode_at, _DeviceContext,
                           _has_global_hook, _transforms, _has_storage))

MAX_LORA_RANK = 8
MAX_LAYERS = 20          # of one linear_group, linear_tiled or expert_combine launch


# The kernels of csrc/moe.hip spend few launches on little work: a tile is 32 x 32 whatever the shape, weights and
# inputs come from L2 without an LDS tile, and some of them are one block.  Where a call is more than that the library's
# kernels win, and these rules end the native form.  Times in us, a pass among others, native / torch.

def router_pays(T: int, H: int, E: int) -> bool:
    """AdaptiveRouter of T tokens.  Inside both the pass and its kernels are faster: 128 x 256, 4 experts 106 / 377; 1024 x 1024,
    64 experts 268 / 416 (kernels 266 / 284); 8192 x 128, 16 experts 130 / 422; 128 x 2048, 8 experts 204 / 435 (kernels 201 / 208).
    Outside: 2048 x 1024, 64 experts 394 / 380; 8192 x 512, 8 experts 310 / 375 with 311 / 288 of kernels; 1024 x 2048 464 / 416;
    16 x 4096 493 / 413 (the selector's weights go through one block); 65536 x 128, 64 experts 5228 / 439 (the balance loss
    is one block)."""
    if H <= 1024:
        return T * H <= 1 << 20 and T * E <= 1 << 17
    return H <= 2048 and T <= 128 and E <= 8


def projections_pay(T: int, H: int, N: int) -> bool:
    """q, k and v of T tokens, N columns in all: 8 x 1024 x 3072 23 / 61, 64 x 2048 x 6144 37 / 60, 8 x 2560 x 7680 25 / 60,
    32 x 3584 x 5376 35 / 62; outside 64 x 3072 x 9216 75 / 61, 8 x 4096 x 12288 51 / 61 with 47 / 41 in a replayed graph,
    64 x 4096 x 12288 101 / 69, 8 x 8192 x 12288 140 / 100; 128 tokens of 2048 x 6144 55 / 59."""
    return T <= 64 and H <= 3584 and H * N <= (20_000_000 if T <= 32 else 13_000_000)


_TILES = ((128, 128, 57.0), (64, 128, 30.0), (64, 64, 16.6), (32, 64, 11.0))   # rows, columns, ns for a round of 256 and a k-value


@lru_cache(maxsize=1024)      # (5 us a call otherwise; a program has a few sizes)
def _tiled_us(T: int, H: int, widths: tuple) -> float:
    """Kernel time of linear_tiled without its start of about 5 us (tile_variant in csrc/linear.hip)."""
    return 1e-3 * H * min(-(-(-(-T // m) * sum(-(-w // n) for w in widths)) // 256) * ns for m, n, ns in _TILES)


def tiled_pays(T: int, H: int, widths) -> bool:
    """The same for 256 tokens and more, in LDS tiles (csrc/linear.hip).  Up to 3.5e9 multiply-adds the library's three calls are
    bound by the host, 57 us: faster while the tiles take less (250 x 512 x 2048 9 / 56, 1000 x 512 x 2048 21 / 56, 500 x 1536 x 4096 52 / 66,
    291 x 1792 x 4096 59 / 61), behind that where they fill their rounds (100 TFLOP/s by the rule: 295 x 3840 x 3072 67 / 85, 397 x 2048 x 4096
    68 / 74; below it 330 x 3072 x 3072 97 / 73, 539 x 3072 x 2048 96 / 83, 639 x 2304 x 2304 74 / 66, 261 x 2048 x 4608 67 / 61).  Beyond 3.5e9
    one round of 128 x 128 tiles that fills the chip: 1280 x 2048 x 3072 125 / 144, 640 x 3072 x 6144 183 / 203, 1792 x 2560 x 2304 155 / 180,
    896 x 3840 x 4608 229 / 267, 1000 x 2048 x 4096 125 / 130, 1024 x 4096 x 4096 245 / 244; below 87 % of it 871 x 3072 x 4096 183 / 177, outside
    4000 x 3072 x 3072 537 / 528.  Of 171 sizes none that it takes was slower by more than half a percent.  Fewer than 256 tokens would be
    faster too (130 x 1024 x 3072 32 / 57), but there the library sums in another order for most widths, and 2e-7 of a query is 1e-5 of a
    probability where scores reach 100; from 256 on it was the same order, to the last bit, for nine of ten sizes measured (nearly all
    others have layers of 256 columns, which the library splits along k)."""
    if T < 256:
        return False
    N = sum(widths)
    if T * H * N <= 3_500_000_000:
        us = _tiled_us(T, H, tuple(widths))
        return us <= 55 or 2e-6 * T * H * N >= 100 * us
    tiles = -(-T // 128) * sum(-(-n // 128) for n in widths)
    return tiles <= 256 and T * N >= 0.87 * 256 * 128 * 128


def experts_tiled(T: int, H: int, E: int) -> bool:
    """The products of E experts [H, H] in one launch of LDS tiles: 128 x 256, 4 experts 14 us for four library calls of 34 on one
    compute unit each, 1053 x 512, 4 experts 32 / 75, 667 x 1024, 4 experts 60 / 76; while the tiles take less time than the
    library's calls take the host, 18 us each (outside 743 x 1536, 1 expert 52 / 36, 716 x 1536, 2 experts 84 / 71, 548 x 1280,
    3 experts 70 / 62).

    What the experts put out is cached in codes, and the means of the caches come back in the next call, where another order of sums
    - 2e-7, a code in 10^4 - grows to 1e-4 of a cached row's scale.  So only sizes are taken where the library (of ROCm 7, as torch
    calls it by default) was measured to sum in the same order, to the last bit: 33 tokens on but for 257 to 1024 and more
    than 2048 tokens of 256 columns, 257 on of 128, and fewer than 512 of more than 512; 2800 sizes up to 8192 tokens, of which 3
    differed, all beyond what the time admits.  Another library or version may choose otherwise: no less exact, but
    its two forms then differ by that much."""
    same_order = (33 <= T <= 8192 and (T <= 256 or H >= 384 or H == 256 and 1024 < T <= 2048) and (H <= 512 or T >= 512))
    return same_order and T * H * H * E <= 3_500_000_000 and _tiled_us(T, H, (H,) * E) <= 18 * E - 6


def key_projection_pays(T: int, H: int) -> bool:
    """One [H, H] layer with LoRA: 1024 x 512 22 / 71, 2048 x 512 34 / 69, 256 x 1024 23 / 74, 128 x 2048 38 / 71; outside
    8192 x 512 111 / 79, 2048 x 1024 90 / 79, 512 x 2048 91 / 71, 128 x 4096 105 / 89."""
    return H <= 512 and T * H <= 1 << 20 or H <= 2048 and T * H <= 1 << 18


def _no_hooks(m: nn.Module) -> bool:
    return not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                or "forward" in m.__dict__)


def plain(m, cls) -> bool:
    """m is exactly a `cls`, and calling it runs that class's forward and nothing else."""
    return type(m) is cls and _no_hooks(m)


def _watched() -> bool:
    """A function or dispatch mode (make_fx, a user's) sees torch's calls; to it the output of a kernel launched beside them is a
    constant.  A default device is a function mode too, but one that only places new tensors."""
    if _dispatch_modes() or _pre_dispatch_modes():
        return True
    n = _function_modes()
    return n > 0 and any(type(_function_mode_at(i)) is not _DeviceContext for i in range(n))


def ordinary_call() -> bool:
    # (is_compiling comes first: what follows it would break a compiled graph)
    return _KNOWN and not (_is_compiling() or _watched() or _has_global_hook() or _is_autocast("cuda") or _is_tracing()
                           or forward_ad._current_level >= 0 or _transforms() is not None)


def ordinary_tensor(t, device, dtype=torch.float32, align: int = 16) -> bool:
    """A dense tensor a kernel may read by its address, `align` bytes at a time (csrc/call.cpp)."""
    return ops.ordinary_tensor(t, device, dtype, align)


def forward_only(x) -> bool:
    """A float32 GPU input of a pass that records nothing."""
    return not torch.is_grad_enabled() and x.is_cuda and ordinary_call() and ordinary_tensor(x, x.device)


def tensors_of(m, a: str, b: str):
    """m.<a>, m.<b>: parameters (the attributes themselves look through three tables for them), buffers or plain attributes."""
    p = m._parameters
    ta, tb = p.get(a), p.get(b)
    return (ta, tb) if ta is not None and tb is not None else (getattr(m, a, None), getattr(m, b, None))


def linear_ok(m, n_in: int, n_out: int, device) -> bool:
    """A plain nn.Linear of this shape with a bias, as linear_group reads it."""
    if not plain(m, nn.Linear):
        return False
    w, b = tensors_of(m, "weight", "bias")
    return (w is not None and b is not None and w.shape == (n_out, n_in) and ordinary_tensor(w, device)
            and ordinary_tensor(b, device))


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
