"""Tensor-level operators over the C ABI of libpikv_hip.so.

Every function validates device / dtype / contiguity / shape in Python, raises
ValueError on a bad argument, allocates the outputs with torch (device memory
and streams are the only things torch is used for here) and enqueues the HIP
kernels on torch's current stream.  There is no CPU path: a CPU tensor is an
error, and a missing library raises PiKVNativeError.

The operator set follows the reference's PiKVKernels facade
(core/single/pikv_kernels.py: top_k_routing :54-99, compress_kv :101-287,
evict_cache :289-422) and the module functions it would have served:
router tail (core/single/pikv_routing.py:65-82), quantise formula
(core/single/module/pikv_compression.py:945-1012), manager append / evict /
compact (core/single/cache_scheduling.py:391-436), H2O bookkeeping (:69-99).
"""
from __future__ import annotations

import math
from typing import Optional, Sequence

import torch

from . import _native as N
from ._native import (BF16, EVICT_ALL, EVICT_H2O, EVICT_LRU, F32, Q_I4_ASYM, Q_I4_SYM,
                      Q_I8_ASYM, Q_I8_SYM, SCORE_TILE)

__all__ = [
    "router_fused", "router_tail", "capacity_slots", "quantize_rows", "quant8_minshift",
    "dequantize_rows", "prefill_attend", "fakequant_colblocks", "fakequant_preset", "CachePool", "scheme_bits",
    "Q_I8_SYM", "Q_I8_ASYM", "Q_I4_ASYM", "Q_I4_SYM", "EVICT_H2O", "EVICT_LRU",
]


# --------------------------------------------------------------------------
# helpers
# --------------------------------------------------------------------------

# the raw handle of torch.cuda.current_stream(), without building the stream object (every caller holds a GPU
# tensor, so the runtime is up); by the public way in a version of torch that names the two calls otherwise
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_raw_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream() -> int:
    if _raw_stream is None or _raw_device is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_raw_device())


def _dt(t: torch.Tensor, name: str) -> int:
    if t.dtype == torch.float32:
        return F32
    if t.dtype == torch.bfloat16:
        return BF16
    raise ValueError(f"{name}: dtype must be float32 or bfloat16, got {t.dtype}")


def _refuse(t, name, dtype, ndim):
    """Says what `t` is not (for _need)."""
    if t is None:
        raise ValueError(f"{name} is required")
    if not isinstance(t, torch.Tensor):
        raise ValueError(f"{name} must be a torch.Tensor")
    if not t.is_cuda:
        raise ValueError(f"{name} must live on the GPU (got {t.device}); there is no CPU path")
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")
    if dtype is not None and t.dtype != dtype:
        raise ValueError(f"{name}: dtype must be {dtype}, got {t.dtype}")
    raise ValueError(f"{name}: expected {ndim} dimensions, got {tuple(t.shape)}")


def _need(*a, **k):
    """_need(t, name, *, dtype=None, ndim=None, optional=False): t, if it is a contiguous GPU tensor of that dtype and
    number of dimensions (or None where that may be); in csrc/call.cpp."""
    N.entry_module()


def ordinary_tensor(*a):
    """ordinary_tensor(t, device, dtype, align): whether t is a dense tensor of that device and dtype that a kernel may read by
    its address, `align` bytes at a time; in csrc/call.cpp."""
    N.entry_module()


if N._call is not None:
    N._call.setup(torch.Tensor, torch.nn.Parameter, _refuse, torch._C._has_storage if hasattr(torch._C, "_has_storage") else bool)
    _need, ordinary_tensor = N._call.need, N._call.ordinary


def _vecf(t, name, n, device):
    """Optional float32 [n] vector on `device`."""
    if t is None:
        return None
    t = torch.as_tensor(t, dtype=torch.float32, device=device).contiguous()
    if t.numel() != n:
        raise ValueError(f"{name} must have {n} elements, got {t.numel()}")
    return t


def scheme_bits(scheme: int) -> int:
    return 8 if scheme in (Q_I8_SYM, Q_I8_ASYM) else 4


def _scheme_asym(scheme: int) -> bool:
    return scheme in (Q_I8_ASYM, Q_I4_ASYM)


def _check_scheme(scheme, D, group):
    if scheme not in (Q_I8_SYM, Q_I8_ASYM, Q_I4_ASYM, Q_I4_SYM):
        raise ValueError(f"unknown quantisation scheme {scheme}")
    epl = 16 if scheme_bits(scheme) == 8 else 32
    if D <= 0 or group <= 0 or D % group:
        raise ValueError(f"group {group} must divide the row width {D}")
    if group & (group - 1) or group < epl or group > 64 * epl:
        raise ValueError(
            f"group must be a power of two in [{epl}, {64 * epl}] for {scheme_bits(scheme)}-bit codes, got {group}")


def _meta_dtype(scheme):
    return torch.float32 if scheme_bits(scheme) == 8 else torch.float16


def _code_plane(rows, D, scheme, device):
    if scheme_bits(scheme) == 8:
        dt = torch.int8 if scheme == Q_I8_SYM else torch.uint8
        return torch.zeros(rows, D, dtype=dt, device=device)
    return torch.zeros(rows, D // 2, dtype=torch.uint8, device=device)


# --------------------------------------------------------------------------
# K1 router
# --------------------------------------------------------------------------

class RouterOut:
    """Compact routing result.  probs [T,E] f32, topk_idx [T,k] i32,
    topk_w [T,k] f32, slot [T,k] i32 (-1 = dropped by capacity) or None,
    count [E] i32 or None, logits [T,E] f32 or None."""
    __slots__ = ("probs", "topk_idx", "topk_w", "slot", "count", "logits", "capacity")

    def __init__(self, probs, topk_idx, topk_w, slot, count, logits, capacity):
        self.probs, self.topk_idx, self.topk_w = probs, topk_idx, topk_w
        self.slot, self.count, self.logits, self.capacity = slot, count, logits, capacity

    @property
    def keep(self):
        return None if self.slot is None else self.slot >= 0


def _router_common(T, E, k, capacity, device, want_probs=True, want_logits=False):
    if not (1 <= E <= 64):
        raise ValueError(f"num_experts must be in [1,64], got {E}")
    if not (1 <= k <= min(E, 8)):
        raise ValueError(f"top_k must be in [1,min(E,8)], got {k}")
    probs = torch.empty(T, E, dtype=torch.float32, device=device) if want_probs else None
    logits = torch.empty(T, E, dtype=torch.float32, device=device) if want_logits else None
    idx = torch.empty(T, k, dtype=torch.int32, device=device)
    w = torch.empty(T, k, dtype=torch.float32, device=device)
    slot = count = ws = None
    ws_bytes = 0
    if capacity is not None:
        if capacity < 0:
            raise ValueError("capacity must be >= 0")
        slot = torch.empty(T, k, dtype=torch.int32, device=device)
        count = torch.empty(E, dtype=torch.int32, device=device)
        ws_bytes = N.size("pikv_router_workspace_bytes", T, E, k)
        ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=device)
    return probs, logits, idx, w, slot, count, ws, ws_bytes


ROUTER_SINGLE, ROUTER_MODULE = 0, 1


def _arith(module_arithmetic: bool) -> int:
    return ROUTER_MODULE if module_arithmetic else ROUTER_SINGLE


def router_fused(x, weight, bias=None, *, top_k=2, capacity=None, expert_scale=None,
                 expert_mask=None, temperature=1.0, renorm_eps=0.0,
                 return_logits=False, module_arithmetic=False) -> RouterOut:
    """Gate projection + softmax + top-k + renormalise (+ capacity slots).
    x [T,H] f32|bf16, weight [E,H] same dtype (nn.Linear layout).
    module_arithmetic=True: the operation order and mask penalty of the reference's
    module/ copy (* expert_scale before / temperature, finfo.min instead of -1e9;
    core/single/module/pikv_routing.py:596-600, :133-134)."""
    x = _need(x, "x", ndim=2)
    weight = _need(weight, "weight", ndim=2)
    if x.dtype != weight.dtype:
        raise ValueError(f"x and weight must share a dtype ({x.dtype} vs {weight.dtype})")
    dt = _dt(x, "x")
    T, H = x.shape
    E = weight.shape[0]
    if weight.shape[1] != H:
        raise ValueError(f"weight must be [E,{H}], got {tuple(weight.shape)}")
    if H % 8:
        raise ValueError(f"hidden size must be a multiple of 8, got {H}")
    dev = x.device
    bias = _vecf(bias, "bias", E, dev)
    expert_scale = _vecf(expert_scale, "expert_scale", E, dev)
    expert_mask = _vecf(expert_mask, "expert_mask", E, dev)
    probs, logits, idx, w, slot, count, ws, ws_bytes = _router_common(
        T, E, top_k, capacity, dev, True, return_logits)
    ws_bytes = N.size("pikv_router_fused_workspace_bytes", T, H, E, top_k)
    ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=dev)
    if T == 0:  # nothing to route (empty tensors have no device address)
        if count is not None:
            count.zero_()
        return RouterOut(probs, idx, w, slot, count, logits, capacity)
    N.launch("pikv_router_fused", x, weight, dt, bias, expert_scale,
             expert_mask, float(temperature), float(renorm_eps), _arith(module_arithmetic),
             T, H, E, top_k,
             int(capacity or 0), probs, logits, idx, w, slot,
             count, ws, ws_bytes, _stream())
    return RouterOut(probs, idx, w, slot, count, logits, capacity)


def router_tail(logits, *, top_k=2, capacity=None, logits_b=None, select=None,
                expert_scale=None, expert_mask=None, temperature=1.0, renorm_eps=0.0,
                use_softmax=True, module_arithmetic=False) -> RouterOut:
    """Router tail on precomputed float32 logits [T,E]."""
    logits = _need(logits, "logits", dtype=torch.float32, ndim=2)
    T, E = logits.shape
    dev = logits.device
    if (logits_b is None) != (select is None):
        raise ValueError("logits_b and select must be given together")
    if logits_b is not None:
        logits_b = _need(logits_b, "logits_b", dtype=torch.float32, ndim=2)
        if logits_b.shape != logits.shape:
            raise ValueError("logits_b must match logits")
        select = _need(select.reshape(-1).to(torch.uint8).contiguous(), "select")
        if select.numel() != T:
            raise ValueError(f"select must have {T} elements")
    expert_scale = _vecf(expert_scale, "expert_scale", E, dev)
    expert_mask = _vecf(expert_mask, "expert_mask", E, dev)
    probs, _, idx, w, slot, count, ws, ws_bytes = _router_common(
        T, E, top_k, capacity, dev, bool(use_softmax), False)
    if T == 0:
        if count is not None:
            count.zero_()
        return RouterOut(probs, idx, w, slot, count, None, capacity)
    N.launch("pikv_router_tail", logits, logits_b, select, expert_scale,
             expert_mask, float(temperature), float(renorm_eps), int(bool(use_softmax)),
             _arith(module_arithmetic), T, E, top_k, int(capacity or 0), probs, idx, w, slot,
             count, ws, ws_bytes, _stream())
    return RouterOut(probs, idx, w, slot, count, None, capacity)


def capacity_slots(expert_idx, num_experts: int, capacity: int):
    """slot / count for expert indices in token-major order."""
    expert_idx = _need(expert_idx, "expert_idx", dtype=torch.int32)
    if not (1 <= num_experts <= 64):
        raise ValueError("num_experts must be in [1,64]")
    if capacity < 0:
        raise ValueError("capacity must be >= 0")
    A = expert_idx.numel()
    dev = expert_idx.device
    slot = torch.empty_like(expert_idx)
    count = torch.empty(num_experts, dtype=torch.int32, device=dev)
    ws_bytes = N.size("pikv_router_workspace_bytes", A, num_experts, 1)
    ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=dev)
    if A == 0:
        return slot, count.zero_()
    N.launch("pikv_capacity_slots", expert_idx, A, num_experts, int(capacity), slot,
             count, ws, ws_bytes, _stream())
    return slot, count


# --------------------------------------------------------------------------
# K2 / K3 on plain rows
# --------------------------------------------------------------------------

def quantize_rows(x, group: int, scheme: int):
    """Quantise x [n,D] per `group` contiguous elements.  Returns
    (codes, scale, zero|None); 4-bit codes are packed two per byte."""
    x = _need(x, "x", ndim=2)
    dt = _dt(x, "x")
    n, D = x.shape
    _check_scheme(scheme, D, group)
    dev = x.device
    codes = _code_plane(n, D, scheme, dev)
    scale = torch.empty(n, D // group, dtype=_meta_dtype(scheme), device=dev)
    zero = torch.empty_like(scale) if _scheme_asym(scheme) else None
    if n == 0:
        return codes, scale, zero
    N.launch("pikv_quantize_rows", x, dt, n, D, group, scheme, 0, codes, scale,
             zero, _stream())
    return codes, scale, zero


def quant8_minshift(x, want_dq: bool = True):
    """Min-shift 8-bit quantisation of whole rows (core/single/pikv_kernels.py:215-232).
    x [n, D] float32 or bfloat16.  Returns (dq float32 [n,D] or None, codes uint8 [n,D],
    scale [n,1], row_min [n,1])."""
    x = _need(x, "x", ndim=2)
    dt = _dt(x, "x")
    n, D = x.shape
    if D < 1:
        raise ValueError("rows must not be empty")
    dev = x.device
    codes = torch.empty(n, D, dtype=torch.uint8, device=dev)
    dq = torch.empty(n, D, dtype=torch.float32, device=dev) if want_dq else None
    scale = torch.empty(n, 1, dtype=torch.float32, device=dev)
    mn = torch.empty(n, 1, dtype=torch.float32, device=dev)
    if n:
        N.launch("pikv_quant8_minshift", x, dt, n, D, codes, dq, scale, mn, _stream())
    return dq, codes, scale, mn


def dequantize_rows(codes, scale, zero, group: int, scheme: int, out_dtype=torch.float32,
                    rows: Optional[torch.Tensor] = None, row0: int = 0, n: Optional[int] = None):
    """(q - zero) * scale for rows `rows` (int64 indices) or [row0, row0+n)."""
    codes = _need(codes, "codes", ndim=2)
    scale = _need(scale, "scale", ndim=2)
    bits = scheme_bits(scheme)
    D = codes.shape[1] * (1 if bits == 8 else 2)
    _check_scheme(scheme, D, group)
    if _scheme_asym(scheme):
        zero = _need(zero, "zero", ndim=2)
    if scale.dtype != _meta_dtype(scheme) or scale.shape != (codes.shape[0], D // group):
        raise ValueError("scale plane has the wrong dtype or shape")
    total = codes.shape[0]
    if rows is not None:
        rows = _need(rows, "rows", dtype=torch.int64, ndim=1)
        cnt = rows.numel()
    else:
        cnt = total - row0 if n is None else n
        if row0 < 0 or cnt < 0 or row0 + cnt > total:
            raise ValueError("row range outside the plane")
    if out_dtype not in (torch.float32, torch.bfloat16):
        raise ValueError("out_dtype must be float32 or bfloat16")
    out = torch.empty(cnt, D, dtype=out_dtype, device=codes.device)
    if cnt == 0:
        return out
    N.launch("pikv_gather_dequant", codes, scale, zero, D, group, scheme,
             rows, row0, cnt, out, F32 if out_dtype == torch.float32 else BF16,
             _stream())
    return out


def fakequant_colblocks(x, group: int, bits: int = 8, symmetric: bool = False):
    """Reference-domain fake quantisation (min/max over all rows x `group`
    columns).  x [N,H] f32 -> (dq [N,H] f32, stats [nblk,4], mse [nblk])."""
    x = _need(x, "x", dtype=torch.float32, ndim=2)
    Nr, H = x.shape
    if group < 1:
        raise ValueError("group must be >= 1")
    nblk = (H + group - 1) // group
    dev = x.device
    out = torch.empty_like(x)
    stats = torch.zeros(nblk, 4, dtype=torch.float32, device=dev)
    mse = torch.zeros(nblk, dtype=torch.float32, device=dev)
    ws_bytes = N.size("pikv_fakequant_workspace_bytes", Nr, H, group)
    ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=dev)
    N.launch("pikv_fakequant_colblocks", x, Nr, H, group, bits, int(bool(symmetric)),
             out, stats, mse, ws, ws_bytes, _stream())
    return out, stats, mse


def fakequant_preset(x, preset, group: int, bits: int = 8, symmetric: bool = False):
    """Fake quantisation with parameters fixed beforehand: `preset` is a (min, max, scale,
    zero) row of a fakequant_colblocks `stats` output; one (scale, zero) serves every
    element.  x [N,H] f32 -> (dq [N,H] f32, mse [nblk] per block of `group` columns)."""
    x = _need(x, "x", dtype=torch.float32, ndim=2)
    preset = _need(preset, "preset", dtype=torch.float32)
    if preset.numel() != 4:
        raise ValueError("preset must hold (min, max, scale, zero)")
    Nr, H = x.shape
    if group < 1:
        raise ValueError("group must be >= 1")
    nblk = (H + group - 1) // group
    dev = x.device
    out = torch.empty_like(x)
    mse = torch.zeros(nblk, dtype=torch.float32, device=dev)
    ws_bytes = N.size("pikv_fakequant_workspace_bytes", Nr, H, group)
    ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=dev)
    N.launch("pikv_fakequant_preset", x, Nr, H, group, bits, int(bool(symmetric)),
             preset, out, mse, ws, ws_bytes, _stream())
    return out, mse


# --------------------------------------------------------------------------
# cache pool
# --------------------------------------------------------------------------

def _evict_workspace(n_caches: int, max_len: int, device):
    nbytes = N.size("pikv_evict_workspace_bytes", n_caches, max_len)
    return torch.empty(max(nbytes, 256), dtype=torch.uint8, device=device), nbytes


def select_top_rows(score, seg_base, seg_len, n_keep, max_len: Optional[int] = None):
    """Per segment c of a flat score array (rows seg_base[c] .. +seg_len[c]): keep
    the n_keep[c] largest scores, ties to the lower index.  Returns (keep_flag
    uint8 [rows], keep_index int32 [rows], n_kept int32 [segments]); segment c's
    ascending survivor list sits at keep_index[seg_base[c] : +n_kept[c]]."""
    score = _need(score, "score", dtype=torch.float32, ndim=1)
    seg_base = _need(seg_base, "seg_base", dtype=torch.int64, ndim=1)
    seg_len = _need(seg_len, "seg_len", dtype=torch.int32, ndim=1)
    n_keep = _need(n_keep, "n_keep", dtype=torch.int32, ndim=1)
    n = seg_base.numel()
    if seg_len.numel() != n or n_keep.numel() != n:
        raise ValueError("seg_base, seg_len and n_keep must have the same length")
    dev = score.device
    flag = torch.zeros(score.numel(), dtype=torch.uint8, device=dev)
    index = torch.zeros(score.numel(), dtype=torch.int32, device=dev)
    kept = torch.zeros(n, dtype=torch.int32, device=dev)
    if n == 0 or score.numel() == 0:
        return flag, index, kept
    zero = torch.zeros(n, dtype=torch.int32, device=dev)
    if max_len is None:   # an upper bound of every segment length that needs no device read
        max_len = score.numel()
    ws, ws_bytes = _evict_workspace(n, int(max_len), dev)
    # H2O selection with an empty "recent" budget; the score doubles as the (unused) timestamp
    N.launch("pikv_evict_select", EVICT_H2O, score, score, seg_base, seg_len,
             n_keep, zero, n, int(max_len), flag, index, kept, ws,
             ws_bytes, _stream())
    return flag, index, kept


def linear_group(x, layers, rank: int = 0):
    """Linear layers over one input x [T, K] float32 in one launch.  `layers`: dicts of weight [N, K], bias [N],
    out [T, N] and optionally relu, lora_a [K, rank], lora_b [rank, N], scaling.  K a multiple of 128, N of
    32, at most 20 layers, rank at most 8."""
    x = _need(x, "x", dtype=torch.float32, ndim=2)
    T, K = x.shape
    for l in layers:
        N_ = l["weight"].shape[0]
        w, b, o = (_need(l[n], n, dtype=torch.float32) for n in ("weight", "bias", "out"))
        if w.shape != (N_, K) or b.shape != (N_,) or o.shape != (T, N_):
            raise ValueError("a layer's weight, bias or out does not match x")
        if l.get("lora_a") is not None:
            a, bb = _need(l["lora_a"], "lora_a", dtype=torch.float32), _need(l["lora_b"], "lora_b", dtype=torch.float32)
            if a.shape != (K, rank) or bb.shape != (rank, N_):
                raise ValueError("a layer's LoRA does not match its weight and the rank")
        if w.data_ptr() % 16 or x.data_ptr() % 16:
            raise ValueError("x and the weights must be 16-byte aligned")
    if T == 0:
        return
    n = len(layers)
    nb = N.size("pikv_linear_group_workspace_bytes", T, n, rank)
    ws = torch.empty(nb, dtype=torch.uint8, device=x.device) if nb else None
    N.launch("pikv_linear_group", x, T, K, n, [l["weight"] for l in layers],
             [l["bias"] for l in layers], [l["weight"].shape[0] for l in layers],
             [int(bool(l.get("relu"))) for l in layers], rank,
             [l.get("lora_a") for l in layers], [l.get("lora_b") for l in layers],
             [float(l.get("scaling", 0.0)) for l in layers],
             [l["out"] for l in layers], ws, nb, _stream())


def linear_tiled(x, layers):
    """Linear layers over one input x [T, K] float32 in one launch of LDS tiles, for many tokens.  `layers`: (weight [N, K],
    bias [N], out [T, N]) of each, at most 20; K a multiple of 64."""
    x = _need(x, "x", dtype=torch.float32, ndim=2)
    T, K = x.shape
    for l in layers:
        w, b, o = (_need(t, n, dtype=torch.float32) for t, n in zip(l, ("weight", "bias", "out")))
        N_ = w.shape[0]
        if w.shape != (N_, K) or b.shape != (N_,) or o.shape != (T, N_):
            raise ValueError("a layer's weight, bias or out does not match x")
    if T == 0:
        return
    n = len(layers)
    w, b, o = zip(*layers)
    N.launch("pikv_linear_tiled", x, T, K, n, w, b, [t.shape[0] for t in w],
             o, _stream())


def value_lora(mean, lora_a, lora_b, scaling):
    """mean[e] + ((mean[e] lora_a[e]) lora_b[e]) * scaling[e] for mean [E, H] float32 and lists of E."""
    mean = _need(mean, "mean", dtype=torch.float32, ndim=2)
    E, H = mean.shape
    lora_a, lora_b = list(lora_a), list(lora_b)          # (a stacked tensor or a ParameterList, too)
    rank = lora_a[0].shape[1]
    if not len(lora_a) == len(lora_b) == len(scaling) == E:
        raise ValueError("one lora_a, lora_b and scaling per row of mean")
    for a, b in zip(lora_a, lora_b):
        if (_need(a, "lora_a", dtype=torch.float32).shape != (H, rank)
                or _need(b, "lora_b", dtype=torch.float32).shape != (rank, H)):
            raise ValueError("lora_a must be [H, rank], lora_b [rank, H]")
    out = torch.empty_like(mean)
    N.launch("pikv_value_lora", mean, E, H, rank, lora_a, lora_b,
             [float(v) for v in scaling], out, _stream())
    return out


def expert_combine(dense, lora, scaling, add, weights, lora_b=None):
    """(outs [E, T, H], mix [T, H]): outs[e] = relu(dense[e] + lora[e] * scaling[e]) + add[e], mix the sum over e, in
    order, of outs[e][t] * weights[t][e].  dense, lora: lists of E (at most 20) tensors [T, H]; add [E, H]; weights
    [T, E]; float32.  With lora_b (E tensors [rank, H]) lora[e] is [T, rank], and its product with lora_b[e] is taken."""
    dense, lora, lora_b = list(dense), list(lora), None if lora_b is None else list(lora_b)     # (stacked tensors, too)
    E, (T, H) = len(dense), dense[0].shape
    if not 1 <= E == len(lora) == len(scaling) or H % 4:
        raise ValueError("one lora and scaling per expert, and a width that is a multiple of 4")
    rank = H if lora_b is None else lora_b[0].shape[0]
    for ts, shape, align in ((dense, (T, H), 16), (lora, (T, rank), 16 if lora_b is None else 4), (lora_b or (), (rank, H), 16)):
        for t in ts:
            if _need(t, "an expert's product", dtype=torch.float32).shape != shape or t.data_ptr() % align:
                raise ValueError(f"the experts' products must be {list(shape)} and {align}-byte aligned")
    if lora_b is not None and len(lora_b) != E:
        raise ValueError("one lora_b per expert")
    add = _need(add, "add", dtype=torch.float32, ndim=2)
    weights = _need(weights, "weights", dtype=torch.float32, ndim=2)
    if add.shape != (E, H) or weights.shape != (T, E) or add.data_ptr() % 16:
        raise ValueError(f"add must be [{E}, {H}], weights [{T}, {E}]")
    outs = torch.empty(E, T, H, dtype=torch.float32, device=add.device)
    mix = torch.empty(T, H, dtype=torch.float32, device=add.device)
    if mix.numel():
        rest = ([float(v) for v in scaling], add, weights, T, E, H, outs, mix, _stream())
        if lora_b is None:
            N.launch("pikv_expert_combine", dense, lora, *rest)
        else:
            N.launch("pikv_expert_combine_factors", dense, lora, lora_b, rank, *rest)
    return outs, mix


def adaptive_router(x_mean, selector, lb, imp, predictor, seq_len: int, top_k: int, mask=None, temp_lb: float = 1.0,
                    temp_imp: float = 1.0, balance_weight: float = 0.01):
    """AdaptiveRouter behind its hidden layers (pikv_adaptive_router).  x_mean [B, H]; selector (w1, b1, w2, b2);
    lb, imp, predictor: (hidden after ReLU [T, .], w, b).  Returns (weights [T, E], idx int64 [T, k], topk_w [T, k],
    balance loss [], importance [T])."""
    x_mean = _need(x_mean, "x_mean", dtype=torch.float32, ndim=2)
    B, H = x_mean.shape
    T, E, H2 = B * seq_len, lb[1].shape[0], predictor[0].shape[1]
    for t, shape in zip((*selector, *lb, *imp, *predictor),
                        ((H2, H), (H2,), (2, H2), (2,), (T, H), (E, H), (E,), (T, H), (E, H), (E,), (T, H2), (1, H2), (1,))):
        if _need(t, "a router tensor", dtype=torch.float32).shape != shape:
            raise ValueError(f"a router tensor has shape {tuple(t.shape)}, expected {shape}")
    if mask is not None and _need(mask, "mask", dtype=torch.float32).shape != (E,):
        raise ValueError("mask must have one value per expert")
    if not (1 <= E <= 64 and 1 <= top_k <= min(E, 8) and T >= 1):
        raise ValueError("num_experts must be in [1,64], top_k in [1,min(E,8)], with at least one token")
    dev = x_mean.device
    blend = torch.empty(B, 2, dtype=torch.float32, device=dev)
    probs = torch.empty(2, T, E, dtype=torch.float32, device=dev)
    idx = torch.empty(T, top_k, dtype=torch.int64, device=dev)
    topk_w = torch.empty(T, top_k, dtype=torch.float32, device=dev)
    importance = torch.empty(T, dtype=torch.float32, device=dev)
    loss = torch.empty((), dtype=torch.float32, device=dev)
    N.launch("pikv_adaptive_router", x_mean, B, seq_len, H, H2, E, top_k, *selector,
             *lb, float(temp_lb), *imp, float(temp_imp),
             *predictor, mask, float(balance_weight), blend, probs[0], probs[1],
             idx, topk_w, importance, loss, _stream())
    return probs[1], idx, topk_w, loss, importance


def prefill_attend(q, k, v, pool: Optional["CachePool"] = None, causal: bool = True,
                   scale_qk: Optional[float] = None):
    """softmax(q.k) v of a prompt chunk in float32: q [B, S, n_q_heads, head_dim] over the rows that
    cache b of `pool` holds (None: nothing cached) and the chunk's own k, v [B, S, n_kv_heads,
    head_dim], query i seeing own rows 0..i (all of them with causal=False).  head_dim 64 or 128.
    Returns out like q."""
    q = _need(q, "q", dtype=torch.float32, ndim=4)
    k = _need(k, "k", dtype=torch.float32, ndim=4)
    v = _need(v, "v", dtype=torch.float32, ndim=4)
    B, S, hq, dh = q.shape
    hkv = k.shape[2]
    if k.shape != (B, S, hkv, dh) or v.shape != k.shape:
        raise ValueError(f"k and v must be [{B}, {S}, kv_heads, {dh}], got {tuple(k.shape)} and {tuple(v.shape)}")
    if hkv == 0 or hq % hkv:
        raise ValueError("the query heads must be a multiple of the kv heads")
    if dh not in (64, 128):
        raise ValueError(f"head_dim must be 64 or 128, got {dh}")
    # the kernel reads 16 bytes at a time: rows that begin elsewhere (a view into a larger buffer) are copied
    q, k, v = (t if t.data_ptr() % 16 == 0 else t.clone() for t in (q, k, v))
    if pool is not None and (pool.n_caches != B or pool.n_heads != hkv or pool.head_dim != dh or not pool.with_v):
        raise ValueError("the pool's caches do not match k and v")
    out = torch.empty_like(q)
    if out.numel() == 0:
        return out
    max_cached = pool.max_cap if pool is not None and pool.rows > 0 else 0
    planes = [None] * 6 if max_cached == 0 else [*pool._planes("k"), *pool._planes("v")]
    nb = N.size("pikv_prefill_attend_workspace_bytes", B, S, hkv, hq, dh, max_cached)
    ws = torch.empty(nb, dtype=torch.uint8, device=q.device) if nb else None
    N.launch("pikv_prefill_attend", q, k, v, B, S, hkv, hq, dh, int(bool(causal)),
             float(1.0 / math.sqrt(dh) if scale_qk is None else scale_qk), *planes,
             pool.scheme if max_cached else Q_I8_SYM, pool.group if max_cached else 0,
             pool.row_base if max_cached else None, pool.fill if max_cached else None, max_cached,
             out, ws, nb, _stream())
    return out


class CachePool:
    """n_caches quantised KV caches (one per expert or per sequence) sharing a
    row space in HBM; see include/pikv_hip.h for the plane layout.  State
    (planes, fill) lives on the GPU; no method reads it back to the host."""

    def __init__(self, caps: Sequence[int], n_heads: int, head_dim: int, group: int,
                 scheme: int, device, with_v: bool = True):
        self.device = torch.device(device)
        if self.device.type != "cuda":
            raise ValueError("CachePool needs a GPU device; there is no CPU path")
        self.n_heads, self.head_dim = int(n_heads), int(head_dim)
        self.D = self.n_heads * self.head_dim
        self.group, self.scheme, self.with_v = int(group), int(scheme), bool(with_v)
        _check_scheme(scheme, self.D, group)
        caps = [int(c) for c in caps]
        if not caps or min(caps) < 0:
            raise ValueError("caps must be a non-empty list of non-negative sizes")
        self.n_caches = len(caps)
        self.max_cap = max(caps)
        base, run = [], 0
        for c in caps:
            base.append(run)
            run += c
        self.rows = run
        self.caps_host, self.base_host = caps, base     # the geometry, for host-side slicing
        dev = self.device
        self.cap = torch.tensor(caps, dtype=torch.int32, device=dev)
        self.row_base = torch.tensor(base, dtype=torch.int64, device=dev)
        self.fill = torch.zeros(self.n_caches, dtype=torch.int32, device=dev)
        ng = self.D // group
        md = _meta_dtype(scheme)
        asym = _scheme_asym(scheme)
        self.k_codes = _code_plane(self.rows, self.D, scheme, dev)
        self.k_scale = torch.zeros(self.rows, ng, dtype=md, device=dev)
        self.k_zero = torch.zeros(self.rows, ng, dtype=md, device=dev) if asym else None
        self.v_codes = self.v_scale = self.v_zero = None
        if with_v:
            self.v_codes = _code_plane(self.rows, self.D, scheme, dev)
            self.v_scale = torch.zeros(self.rows, ng, dtype=md, device=dev)
            self.v_zero = torch.zeros(self.rows, ng, dtype=md, device=dev) if asym else None
        self.acc = torch.zeros(self.rows, dtype=torch.float32, device=dev)
        self.ts = torch.zeros(self.rows, dtype=torch.float32, device=dev)
        # eviction scratch
        self.keep_flag = torch.zeros(self.rows, dtype=torch.uint8, device=dev)
        self.keep_index = torch.zeros(self.rows, dtype=torch.int32, device=dev)
        self.new_len = torch.zeros(self.n_caches, dtype=torch.int32, device=dev)
        self.n_heavy = torch.zeros(self.n_caches, dtype=torch.int32, device=dev)
        self.n_recent = torch.zeros(self.n_caches, dtype=torch.int32, device=dev)
        self._budgets = torch.empty(3 * self.n_caches, dtype=torch.int32, device=dev)
        self._row_bytes = self._plane_row_bytes()

    def _plane_row_bytes(self):
        return [math.prod(p.shape[1:]) * p.element_size() for p in self.planes()]

    def __setstate__(self, state):
        """A copied or unpickled pool makes its workspaces anew: their sizes, and what else is derived from the planes, are those
        of the version that made it."""
        self.__dict__.update((k, v) for k, v in state.items() if k not in ("_decode_ws", "_decode_ws_key", "_evict_ws"))
        self._row_bytes = self._plane_row_bytes()

    # ---- checkpoint ----
    _STATE_PLANES = ("k_codes", "k_scale", "k_zero", "v_codes", "v_scale", "v_zero", "acc", "ts")

    def state_dict(self, trim: bool = True):
        """Everything needed to restore the caches: geometry, fill counts and the
        quantised planes (codes, scales, zero points, accumulators, timestamps) as
        CPU tensors.  With trim=True only the valid rows of every cache are kept
        (rows [row_base[c], row_base[c]+fill[c]), concatenated in cache order)."""
        fill = self.fill.cpu()
        sd = {"layout": torch.tensor([self.n_heads, self.head_dim, self.group, self.scheme,
                                      int(self.with_v), int(trim)], dtype=torch.int64),
              "cap": self.cap.cpu(), "fill": fill}
        rows = None
        if trim:
            base = self.row_base.cpu()
            rows = torch.cat([torch.arange(int(base[c]), int(base[c]) + int(fill[c]))
                              for c in range(self.n_caches)]) if self.n_caches else torch.zeros(0, dtype=torch.int64)
            rows = rows.to(self.device)
        for name in self._STATE_PLANES:
            t = getattr(self, name)
            if t is not None:
                sd[name] = (t.index_select(0, rows) if rows is not None else t).cpu()
        return sd

    def load_state_dict(self, sd):
        """Restore what state_dict() saved into a pool of the same geometry."""
        layout = [int(v) for v in sd["layout"]]
        mine = [self.n_heads, self.head_dim, self.group, self.scheme, int(self.with_v)]
        if layout[:5] != mine:
            raise ValueError(f"checkpoint layout {layout[:5]} does not match this pool {mine}")
        if not torch.equal(sd["cap"].to(torch.int32).cpu(), self.cap.cpu()):
            raise ValueError("checkpoint cache capacities do not match this pool")
        fill = sd["fill"].to(torch.int32)
        if bool((fill > self.cap.cpu()).any()) or bool((fill < 0).any()):
            raise ValueError("checkpoint fill counts exceed the capacities")
        trim = bool(layout[5])
        rows = None
        if trim:
            base = self.row_base.cpu()
            rows = torch.cat([torch.arange(int(base[c]), int(base[c]) + int(fill[c]))
                              for c in range(self.n_caches)]).to(self.device)
        for name in self._STATE_PLANES:
            t = getattr(self, name)
            if t is None:
                continue
            src = sd[name].to(self.device)
            if src.dtype != t.dtype or src.shape[1:] != t.shape[1:]:
                raise ValueError(f"checkpoint plane {name} has the wrong dtype or row shape")
            if rows is not None:
                if src.shape[0] != rows.numel():
                    raise ValueError(f"checkpoint plane {name} does not hold the saved rows")
                t.index_copy_(0, rows, src)
            else:
                if src.shape != t.shape:
                    raise ValueError(f"checkpoint plane {name} has the wrong number of rows")
                t.copy_(src)
        self.fill.copy_(fill.to(self.device))

    # ---- write path ----
    def quant_scatter(self, k_src, v_src, cache_id, slot, fanout: int, now: float = 0.0):
        """Quantise source rows once and append them to their routed caches.
        k_src/v_src [n_src, D] (or [n_src, heads, head_dim]); cache_id/slot
        int32 [n_src*fanout] (any shape).  fill is not advanced."""
        k_src = _need(k_src, "k_src")
        dt = _dt(k_src, "k_src")
        k2 = k_src.reshape(-1, self.D)
        n_src = k2.shape[0]
        v2 = None
        if self.with_v:
            v_src = _need(v_src, "v_src", dtype=k_src.dtype)
            v2 = v_src.reshape(-1, self.D)
            if v2.shape != k2.shape:
                raise ValueError("v_src must match k_src")
        cache_id = _need(cache_id, "cache_id", dtype=torch.int32)
        slot = _need(slot, "slot", dtype=torch.int32)
        if not (1 <= fanout <= 8):
            raise ValueError("fanout must be in [1,8]")
        if cache_id.numel() != n_src * fanout or slot.numel() != n_src * fanout:
            raise ValueError(f"cache_id/slot must have n_src*fanout = {n_src * fanout} elements")
        if n_src == 0:
            return
        N.launch("pikv_quant_scatter", k2, v2, dt, n_src, fanout, self.D, self.group,
                 self.scheme, cache_id, slot, self.row_base, self.fill,
                 self.cap, self.n_caches, self.k_codes, self.v_codes,
                 self.k_scale, self.v_scale, self.k_zero, self.v_zero,
                 self.acc, self.ts, float(now), _stream())

    def quant_scatter_routed(self, k_src, v_src, cache_id, slot, per_token: int, now: float = 0.0):
        """quant_scatter for rows that differ per cache: assignment j of token t (cache_id / slot
        [n_tokens * per_token]) takes the K row k_src[t] and the V row v_src[cache_id][t] of k_src
        [n_tokens, D] and v_src [n_caches, n_tokens, D], float32.  fill is not advanced."""
        if not self.with_v:
            raise ValueError("this pool stores no V rows")
        k_src = _need(k_src, "k_src", dtype=torch.float32, ndim=2)
        n = k_src.shape[0]
        v_src = _need(v_src, "v_src", dtype=torch.float32, ndim=3)
        if k_src.shape[1] != self.D or v_src.shape != (self.n_caches, n, self.D):
            raise ValueError(f"k_src must be [n, {self.D}], v_src [{self.n_caches}, n, {self.D}]")
        cache_id = _need(cache_id, "cache_id", dtype=torch.int32)
        slot = _need(slot, "slot", dtype=torch.int32)
        if not 1 <= per_token <= 64 or cache_id.numel() != n * per_token or slot.numel() != n * per_token:
            raise ValueError("cache_id and slot must have n * per_token elements")
        if n == 0:
            return
        N.launch("pikv_quant_scatter_routed", k_src, v_src, n, per_token, self.D, self.group, self.scheme,
                 cache_id, slot, self.row_base, self.fill, self.cap, self.n_caches,
                 self.k_codes, self.v_codes, self.k_scale, self.v_scale, self.k_zero,
                 self.v_zero, self.acc, self.ts, float(now), _stream())

    def quant_gather(self, k_src, v_src, src_row_base, src_index, n_take, max_take: int,
                     src_score=None, now: float = 0.0):
        """Quantise the listed source rows into the caches in list order: for
        cache c and j < n_take[c], source row src_row_base[c] +
        src_index[src_row_base[c] + j] goes to cache row fill[c] + j.  fill is
        not advanced."""
        k_src = _need(k_src, "k_src")
        dt = _dt(k_src, "k_src")
        k2 = k_src.reshape(-1, self.D)
        v2 = None
        if self.with_v:
            v_src = _need(v_src, "v_src", dtype=k_src.dtype)
            v2 = v_src.reshape(-1, self.D)
            if v2.shape != k2.shape:
                raise ValueError("v_src must match k_src")
        src_row_base = _need(src_row_base, "src_row_base", dtype=torch.int64, ndim=1)
        src_index = _need(src_index, "src_index", dtype=torch.int32, ndim=1)
        n_take = _need(n_take, "n_take", dtype=torch.int32, ndim=1)
        if src_row_base.numel() != self.n_caches or n_take.numel() != self.n_caches:
            raise ValueError("src_row_base / n_take must have one entry per cache")
        if src_index.numel() < k2.shape[0]:
            raise ValueError("src_index must cover the source row space")
        if src_score is not None:
            src_score = _need(src_score, "src_score", dtype=torch.float32)
            if src_score.numel() != k2.shape[0]:
                raise ValueError("src_score must have one entry per source row")
        if max_take <= 0 or k2.shape[0] == 0:
            return
        N.launch("pikv_quant_gather", k2, v2, dt, self.D, self.group, self.scheme,
                 src_row_base, src_index, n_take, int(max_take), src_score,
                 self.row_base, self.fill, self.cap, self.n_caches,
                 self.k_codes, self.v_codes, self.k_scale, self.v_scale,
                 self.k_zero, self.v_zero, self.acc, self.ts, float(now),
                 _stream())

    def advance(self, count, per_call_limit: int = -1):
        """fill[c] = min(fill[c] + min(count[c], limit), cap[c])."""
        count = _need(count, "count", dtype=torch.int32, ndim=1)
        if count.numel() != self.n_caches:
            raise ValueError("count must have one entry per cache")
        N.launch("pikv_cache_advance", self.fill, count, self.cap, self.n_caches,
                 int(per_call_limit), _stream())

    # ---- read path ----
    def _planes(self, which):
        if which == "k":
            return self.k_codes, self.k_scale, self.k_zero
        if which == "v" and self.with_v:
            return self.v_codes, self.v_scale, self.v_zero
        raise ValueError("which must be 'k' or 'v' (and the pool must hold V)")

    def gather_dequant(self, which="k", rows=None, row0=0, n=None, out_dtype=torch.float32):
        codes, scale, zero = self._planes(which)
        return dequantize_rows(codes, scale, zero, self.group, self.scheme, out_dtype,
                               rows=rows, row0=row0, n=n)

    def mean_rows(self, which="v"):
        """Mean dequantised row of every cache, [n_caches, D] float32 (zero for an empty cache)."""
        codes, scale, zero = self._planes(which)
        out = torch.empty(self.n_caches, self.D, dtype=torch.float32, device=self.device)
        if self.rows == 0:
            return out.zero_()
        nb = N.size("pikv_cache_mean_workspace_bytes", self.n_caches, self.D, self.max_cap)
        ws = torch.empty(nb, dtype=torch.uint8, device=self.device)
        N.launch("pikv_cache_mean", codes, scale, zero, self.scheme, self.group, self.D,
                 self.row_base, self.fill, self.n_caches, self.max_cap, out, ws, nb, _stream())
        return out

    def scores(self, q, n_q_heads: int, scale_qk: Optional[float] = None,
               max_len: Optional[int] = None):
        """scores[c,h,n] = q[c,h,:] . dequant(K[c,n,h//rep,:]) * scale_qk for
        n < fill[c].  q [n_caches, n_q_heads, head_dim] f32|bf16.  Returns
        (scores [n_caches,n_q_heads,stride] f32, tile_max, tile_sum)."""
        q = _need(q, "q", ndim=3)
        qdt = _dt(q, "q")
        if q.shape != (self.n_caches, n_q_heads, self.head_dim):
            raise ValueError(f"q must be [{self.n_caches},{n_q_heads},{self.head_dim}]")
        if n_q_heads % self.n_heads:
            raise ValueError("n_q_heads must be a multiple of the kv heads")
        max_len = self.max_cap if max_len is None else int(max_len)
        stride = max_len
        n_tiles = (max_len + SCORE_TILE - 1) // SCORE_TILE
        dev = self.device
        scores = torch.empty(self.n_caches, n_q_heads, stride, dtype=torch.float32, device=dev)
        tmax = torch.empty(self.n_caches, max(n_tiles, 1), n_q_heads, dtype=torch.float32, device=dev)
        tsum = torch.empty_like(tmax)
        if scale_qk is None:
            scale_qk = 1.0 / (self.head_dim ** 0.5)
        N.launch("pikv_gather_dequant_scores", self.k_codes, self.k_scale,
                 self.k_zero, self.scheme, self.group, self.n_heads, n_q_heads, self.head_dim,
                 q, qdt, float(scale_qk), self.row_base, self.fill, self.n_caches,
                 max_len, stride, scores, tmax, tsum, _stream())
        return scores, tmax, tsum

    def h2o_accumulate(self, scores, tile_max, tile_sum, now: float, decay: float = 1.0,
                       write_probs: bool = False, return_importance: bool = False,
                       stats_only: bool = False):
        """Normalise, sum over heads, acc += importance, ts = now.  stats_only=True
        leaves acc and ts alone and only fills self.head_stats (for an attend_values
        call that accumulates itself)."""
        scores = _need(scores, "scores", dtype=torch.float32, ndim=3)
        tile_max = _need(tile_max, "tile_max", dtype=torch.float32, ndim=3)
        tile_sum = _need(tile_sum, "tile_sum", dtype=torch.float32, ndim=3)
        nc, hq, stride = scores.shape
        if nc != self.n_caches:
            raise ValueError("scores must have one slab per cache")
        n_tiles = (stride + SCORE_TILE - 1) // SCORE_TILE
        if tile_max.shape != (nc, max(n_tiles, 1), hq) or tile_sum.shape != tile_max.shape:
            raise ValueError("tile statistics do not match scores")
        dev = self.device
        imp = torch.zeros(nc, stride, dtype=torch.float32, device=dev) if return_importance else None
        head_stats = torch.empty(nc, hq, 2, dtype=torch.float32, device=dev)
        N.launch("pikv_h2o_accumulate", scores, tile_max, tile_sum, hq,
                 self.row_base, self.fill, nc, stride, stride, float(decay), float(now),
                 int(bool(write_probs)), None if stats_only else self.acc,
                 None if stats_only else self.ts, imp, head_stats, _stream())
        self.head_stats = head_stats   # (max, sum) per (cache, head): what attend_values normalises with
        return imp

    def attend_values(self, scores, head_stats=None, accumulate: bool = False, now: float = 0.0,
                      decay: float = 1.0):
        """out[c,h,:] = sum_n p[c,h,n] * dequant(V[c,n,h/rep,:]) over the valid rows.
        scores [n_caches, n_q_heads, stride] float32: raw scores together with
        head_stats [n_caches, n_q_heads, 2] (as left in self.head_stats by
        h2o_accumulate), or probabilities when head_stats is None.
        accumulate=True also does h2o_accumulate's bookkeeping (acc = acc*decay + sum of
        the probabilities over the heads, ts = now) in the same pass."""
        if not self.with_v:
            raise ValueError("this pool stores no V rows")
        scores = _need(scores, "scores", dtype=torch.float32, ndim=3)
        nc, hq, stride = scores.shape
        if nc != self.n_caches or hq % self.n_heads:
            raise ValueError("scores must be [n_caches, n_q_heads, stride] with n_q_heads a multiple of the kv heads")
        if head_stats is not None:
            head_stats = _need(head_stats, "head_stats", dtype=torch.float32, ndim=3)
            if head_stats.shape != (nc, hq, 2):
                raise ValueError("head_stats must be [n_caches, n_q_heads, 2]")
        dev = self.device
        out = torch.zeros(nc, hq, self.head_dim, dtype=torch.float32, device=dev)
        if stride == 0:
            return out
        ws_bytes = N.size("pikv_attend_workspace_bytes", nc, hq, self.head_dim, stride)
        ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=dev)
        N.launch("pikv_attend_values", scores, head_stats, stride, self.v_codes,
                 self.v_scale, self.v_zero, self.scheme, self.group, self.n_heads, hq,
                 self.head_dim, self.row_base, self.fill, nc, stride, float(decay), float(now),
                 self.acc if accumulate else None, self.ts if accumulate else None,
                 out, ws, ws_bytes, _stream())
        return out

    def decode_attend(self, q, n_q_heads: int, now: float = 0.0, scale_qk: Optional[float] = None,
                      max_len: Optional[int] = None, accumulate: bool = True, decay: float = 1.0):
        """The whole decode read in one native call (pikv_decode_attend): scores of q
        [n_caches, n_q_heads, head_dim] against the compressed K rows, softmax over each cache's
        rows, attention output over the compressed V rows -> out [n_caches, n_q_heads, head_dim]
        float32; accumulate=True adds the probabilities to the H2O accumulators (acc = acc*decay +
        sum over the heads, ts = now).  The score matrix stays inside the library's workspace."""
        if not self.with_v:
            raise ValueError("this pool stores no V rows")
        q = _need(q, "q", ndim=3)
        dt = _dt(q, "q")
        if q.shape != (self.n_caches, n_q_heads, self.head_dim):
            raise ValueError(f"q must be [{self.n_caches},{n_q_heads},{self.head_dim}], got {tuple(q.shape)}")
        if n_q_heads % self.n_heads:
            raise ValueError("n_q_heads must be a multiple of the kv heads")
        if scale_qk is None:
            scale_qk = 1.0 / math.sqrt(self.head_dim)
        max_len = self.max_cap if max_len is None else int(max_len)
        dev = self.device
        out = torch.empty(self.n_caches, n_q_heads, self.head_dim, dtype=torch.float32, device=dev)
        key = (n_q_heads, max_len)
        if getattr(self, "_decode_ws_key", None) != key:
            nb = N.size("pikv_decode_attend_workspace_bytes", self.n_caches, n_q_heads, self.head_dim, max_len)
            self._decode_ws = torch.empty(max(nb, 256), dtype=torch.uint8, device=dev)
            self._decode_ws_key = key
        ws = self._decode_ws
        N.launch("pikv_decode_attend", self.k_codes, self.k_scale, self.k_zero,
                 self.v_codes, self.v_scale, self.v_zero, self.scheme, self.group,
                 self.n_heads, n_q_heads, self.head_dim, q, dt, float(scale_qk), self.row_base,
                 self.fill, self.n_caches, max_len, float(decay), float(now),
                 self.acc if accumulate else None, self.ts if accumulate else None,
                 out, ws, ws.numel(), _stream())
        return out

    # ---- eviction ----
    def evict_select(self, policy: int, *, heavy_ratio=0.1, recent_ratio=0.1,
                     n_heavy=None, n_recent=None, n_evict=None, multi_block: bool = True):
        """Fill keep_flag / keep_index / new_len.  H2O: budgets from the
        ratios (per cache, from its current fill) or explicit int32 tensors;
        LRU: n_evict int32 [n_caches].  multi_block=False withholds the workspace, so
        that one block selects each cache whatever its length (same result)."""
        ratios = policy == EVICT_H2O and n_heavy is None
        if ratios:
            nh, nr = self.n_heavy, self.n_recent
        elif policy == EVICT_H2O:
            nh = _need(n_heavy, "n_heavy", dtype=torch.int32, ndim=1)
            nr = _need(n_recent, "n_recent", dtype=torch.int32, ndim=1)
        elif policy == EVICT_LRU:
            nh = _need(n_evict, "n_evict", dtype=torch.int32, ndim=1)
            nr = None
        else:
            raise ValueError(f"unknown eviction policy {policy}")
        if nh.numel() != self.n_caches or (nr is not None and nr.numel() != self.n_caches):
            raise ValueError("budgets must have one entry per cache")
        ws, ws_bytes = None, 0
        if multi_block:
            if getattr(self, "_evict_ws", None) is None:
                self._evict_ws = _evict_workspace(self.n_caches, self.max_cap, self.device)
            ws, ws_bytes = self._evict_ws
        args = (self.acc, self.ts, self.row_base, self.fill, nh, nr, self.n_caches,
                self.max_cap, self.keep_flag, self.keep_index, self.new_len, ws, ws_bytes, _stream())
        if ratios:
            N.launch("pikv_evict_select_h2o", float(heavy_ratio), float(recent_ratio), *args)
        else:
            N.launch("pikv_evict_select", policy, *args)

    def planes(self):
        ps = [self.k_codes, self.k_scale, self.k_zero, self.v_codes, self.v_scale, self.v_zero,
              self.acc, self.ts]
        return [p for p in ps if p is not None]

    def compact(self, extra_planes: Sequence[torch.Tensor] = ()):
        """Move survivors (keep_index/new_len) to the front of every plane and
        set fill = new_len."""
        extra = [_need(p, "extra plane") for p in extra_planes]      # (an iterator gives them once)
        ps = self.planes() + extra
        if len(ps) > N.MAX_PLANES:
            raise ValueError(f"at most {N.MAX_PLANES} planes")
        rbs = self._row_bytes + [math.prod(p.shape[1:]) * p.element_size() for p in extra]
        N.launch("pikv_compact_rows", ps, rbs, len(ps), self.row_base, self.keep_index,
                 self.new_len, self.fill, self.n_caches, _stream())

    def make_room(self, policy: int, *, count: Optional[torch.Tensor] = None, count_all: int = 0,
                  limit: int = -1, heavy_ratio: float = 0.1, recent_ratio: float = 0.1,
                  leave_room: bool = False, append: bool = False):
        """Caches that min(count[c] or count_all, limit, cap[c]) new rows would overflow evict by
        `policy` (EVICT_H2O, EVICT_LRU, EVICT_ALL) and are compacted; the others keep their rows.
        new_len = the rows kept; fill = new_len, or the fill after the new rows with append=True (for an
        append_rows call that is sure to follow: until then the caches claim rows they do not hold)."""
        if count is not None:
            count = _need(count, "count", dtype=torch.int32, ndim=1)
            if count.numel() != self.n_caches:
                raise ValueError("count must have one entry per cache")
        if policy not in (EVICT_H2O, EVICT_LRU, EVICT_ALL):
            raise ValueError(f"unknown eviction policy {policy}")
        ps = self.planes()
        rbs = self._row_bytes
        if getattr(self, "_evict_ws", None) is None:
            self._evict_ws = _evict_workspace(self.n_caches, self.max_cap, self.device)
        ws, ws_bytes = self._evict_ws
        N.launch("pikv_cache_make_room", policy, count, int(count_all), int(limit), float(heavy_ratio),
                 float(recent_ratio), int(leave_room), int(append), self.acc, self.ts, self.row_base,
                 self.fill, self.cap, self.n_caches, self.max_cap, ps, rbs, len(ps), self.keep_flag,
                 self.keep_index, self.new_len, self._budgets, ws, ws_bytes, _stream())

    def append_rows(self, k_src, v_src, now: float = 0.0, advance: bool = False):
        """Quantise k_src / v_src [n_caches * rows, D] (cache-major) behind the new_len rows of every
        cache, as make_room has left them; rows past the capacity are dropped.  advance=True also moves
        fill behind them, in the same launch (after make_room(append=True) it is there already)."""
        k_src = _need(k_src, "k_src")
        dt = _dt(k_src, "k_src")
        rows = k_src.numel() // (self.D * self.n_caches)
        if k_src.numel() != rows * self.D * self.n_caches:
            raise ValueError("k_src must hold the same number of rows for every cache")
        if self.with_v:
            v_src = _need(v_src, "v_src", dtype=k_src.dtype)
            if v_src.numel() != k_src.numel():
                raise ValueError("v_src must match k_src")
        if rows == 0:
            return
        N.launch("pikv_quant_append", k_src, v_src if self.with_v else None, dt, rows, self.D, self.group,
                 self.scheme, self.row_base, self.new_len, self.fill if advance else None, self.cap,
                 self.n_caches, self.k_codes, self.v_codes, self.k_scale, self.v_scale, self.k_zero,
                 self.v_zero, self.acc, self.ts, float(now), _stream())

    def evict(self, policy: int, **kw):
        self.evict_select(policy, **kw)
        self.compact()
