"""GPU parity of the float32 dense kernels of the mixture-of-experts layer, against float64 or the torch path."""
import numpy as np
import pytest

import pikv_oracle as O
from test_gpu_read_evict import _fill_pool
from util import np_of, rng, to_dev

pytestmark = pytest.mark.gpu


def _near(got, want, n, size):
    """A float32 sum of n products of values up to `size`: 2^-24 a step, random signs, four times that."""
    assert np.abs(np_of(got).astype(np.float64) - want).max() <= 4 * 2.0 ** -24 * np.sqrt(n) * size * size


@pytest.mark.parametrize("T,K,widths,rank", [(1, 128, [32], 0), (33, 256, [256, 64, 96], 4), (64, 640, [32, 512], 8),
                                             (500, 128, [64] * 20, 1)])
def test_linear_group(dev, T, K, widths, rank):
    from pikv_amd import ops
    import torch
    r = rng(T + K)
    x = r.standard_normal((T, K)).astype(np.float32)
    layers, want = [], []
    for i, n in enumerate(widths):
        w, b = (r.standard_normal(s).astype(np.float32) for s in ((n, K), (n,)))
        y = x.astype(np.float64) @ w.T.astype(np.float64) + b
        l = dict(weight=to_dev(w, dev), bias=to_dev(b, dev), relu=i % 2 == 0, out=torch.empty(T, n, device=dev))
        if rank and i != 1:
            la, lb = (r.standard_normal(s).astype(np.float32) for s in ((K, rank), (rank, n)))
            y = y + x.astype(np.float64) @ la @ lb.astype(np.float64) * 0.25
            l.update(lora_a=to_dev(la, dev), lora_b=to_dev(lb, dev), scaling=0.25)
        y = np.maximum(y, 0) if l["relu"] else y
        layers.append(l)
        want.append(y)
    ops.linear_group(to_dev(x, dev), layers, rank=rank)
    for l, y in zip(layers, want):
        _near(l["out"], y, K * max(rank, 1), 4.5)


@pytest.mark.parametrize("T,K,widths", [(1, 64, [1]), (31, 64, [65, 3, 64]), (33, 192, [64] * 20), (129, 128, [50257]),   # 32 x 64 tiles, 64 x 64
                                        (256, 64, [4000]), (300, 320, [1000, 1500, 50]),                  # 64 x 64
                                        (511, 128, [2048, 1025, 1000]),                                   # 64 x 128
                                        (1000, 64, [2048, 1024, 1024]), (641, 448, [5000, 130])])         # 128 x 128
def test_linear_tiled(dev, T, K, widths):
    from pikv_amd import ops
    import torch
    r = rng(T + K)
    x = r.standard_normal((T, K)).astype(np.float32)
    layers, want = [], []
    for n in widths:
        w, b = (r.standard_normal(s).astype(np.float32) for s in ((n, K), (n,)))
        want.append(x.astype(np.float64) @ w.T.astype(np.float64) + b)
        # a guard row behind the outputs: a tile's last rows and columns must not be written
        layers.append((to_dev(w, dev), to_dev(b, dev), torch.full((T + 1, n), 7.0, device=dev)))
    ops.linear_tiled(to_dev(x, dev), [(w, b, o[:T]) for w, b, o in layers])
    for (_, _, o), y in zip(layers, want):
        _near(o[:T], y, K, 4.5)
        assert bool((o[T] == 7.0).all())


@pytest.mark.parametrize("E,T,H", [(1, 1, 4), (3, 37, 132), (20, 5, 64)])
def test_expert_combine(dev, E, T, H):
    """Bit for bit what the torch operations give, each rounded on its own (a scaling that is no power of two: a fused
    multiply-add would show), a NaN and infinities among the products."""
    import torch
    from pikv_amd import ops
    torch.manual_seed(E)
    scaling = [0.3 + 0.1 * e for e in range(E)]
    d, l, c, w = (torch.randn(*s, device=dev) for s in ((E, T, H), (E, T, H), (E, H), (T, E)))
    d[0, 0, 0], d[E - 1, T - 1, 1], l[0, 0, 2] = float("nan"), float("inf"), float("-inf")
    outs, mix = ops.expert_combine(list(d), list(l), scaling, c, w)
    want = torch.zeros(T, H, device=dev)
    for e in range(E):
        o = torch.relu(d[e] + l[e] * scaling[e]) + c[e]
        assert torch.equal(o.nan_to_num(7.0), outs[e].nan_to_num(7.0))
        want = want + o * w[:, e:e + 1]
    assert torch.equal(want.nan_to_num(7.0), mix.nan_to_num(7.0))


@pytest.mark.parametrize("E,T,H,rank", [(1, 1, 4, 1), (3, 37, 132, 4), (20, 5, 64, 8)])
def test_expert_combine_factors(dev, E, T, H, rank):
    """Bit for bit the form that is given the products, as torch.mm makes them."""
    import torch
    from pikv_amd import ops
    torch.manual_seed(E)
    scaling = [0.3 + 0.1 * e for e in range(E)]
    d, t, b, c, w = (torch.randn(*s, device=dev) for s in ((E, T, H), (E, T, rank), (E, rank, H), (E, H), (T, E)))
    d[0, 0, 0], t[E - 1, T - 1, 0] = float("nan"), float("inf")
    want = ops.expert_combine(list(d), [torch.mm(x, y) for x, y in zip(t, b)], scaling, c, w)
    got = ops.expert_combine(list(d), list(t), scaling, c, w, lora_b=list(b))
    for g, x in zip(got, want):
        assert torch.equal(g.nan_to_num(7.0), x.nan_to_num(7.0))


@pytest.mark.parametrize("T,H", [(33, 128), (17, 256), (256, 256), (257, 256), (1025, 256), (40, 512), (1000, 512), (700, 1024)])
def test_tiled_experts_sum_in_the_librarys_order(dev, T, H):
    import torch
    from pikv_amd import dense, ops
    torch.manual_seed(T)
    x, w, b = torch.randn(T, H, device=dev), torch.randn(H, H, device=dev) * 0.05, torch.randn(H, device=dev)
    if dense.experts_tiled(T, H, 4):
        o = torch.empty(T, H, device=dev)
        ops.linear_tiled(x, [(w, b, o)])
        assert torch.equal(o, torch.nn.functional.linear(x, w, b))
    else:
        assert (T, H) in ((17, 256), (257, 256))


@pytest.mark.parametrize("H", [128, 256, 384, 512, 640, 1024])
def test_tiled_experts_order_at_the_edges_of_the_rule(dev, H):
    """Both sides of every size where the rule changes, and some between, as many experts as the time admits."""
    import torch
    from pikv_amd import dense, ops
    taken = 0
    for T in (33, 64, 128, 255, 256, 257, 511, 512, 513, 700, 1000, 1023, 1024, 1025, 1500, 2047, 2048, 2049, 3000, 3333, 5000, 8192):
        if not any(dense.experts_tiled(T, H, E) for E in (1, 2, 4)):
            continue
        taken += 1
        torch.manual_seed(T)
        x, w, b = torch.randn(T, H, device=dev), torch.randn(H, H, device=dev) * 0.05, torch.randn(H, device=dev)
        o = torch.empty(T, H, device=dev)
        ops.linear_tiled(x, [(w, b, o)])
        assert torch.equal(o, torch.nn.functional.linear(x, w, b)), T
    assert taken >= 3


@pytest.mark.parametrize("H", [256, 512])
@pytest.mark.parametrize("T", [33, 257, 2048])
def test_expert_factors_sum_in_the_librarys_order(dev, T, H):
    """The second factor at the widths and token counts in use, every rank."""
    import torch
    from pikv_amd import ops
    for rank in range(1, 9):
        torch.manual_seed(T + rank)
        d, t, b, c, w = (torch.randn(*s, device=dev) for s in ((2, T, H), (2, T, rank), (2, rank, H), (2, H), (T, 2)))
        want = ops.expert_combine(list(d), [torch.mm(x, y) for x, y in zip(t, b)], [0.3, 0.7], c, w)
        got = ops.expert_combine(list(d), list(t), [0.3, 0.7], c, w, lora_b=list(b))
        assert all(torch.equal(x, y) for x, y in zip(got, want)), rank


@pytest.mark.parametrize("scheme,D,group", [(O.Q_I8_SYM, 272, 16), (O.Q_I8_ASYM, 256, 256), (O.Q_I4_ASYM, 1088, 32),
                                            (O.Q_I4_SYM, 64, 64)])
@pytest.mark.parametrize("lens", [[0, 1, 63], [65, 64, 130], [5000, 4097, 2]])
def test_mean_rows(dev, scheme, D, group, lens):
    pool, ref = _fill_pool(dev, rng(D + lens[0]), [max(lens)] * 3, lens, 1, D, group, scheme)
    got = np_of(pool.mean_rows("v")).astype(np.float64)
    for c, n in enumerate(lens):
        rows = ref.valid_rows(c)[:n]
        v = O.dequantize_groups(ref.v_codes[rows], ref.v_scale[rows], ref.v_zero[rows], group).astype(np.float64)
        want = v.mean(axis=0) if n else np.zeros(D)
        assert np.abs(got[c] - want).max() <= 4 * 2.0 ** -24 * np.sqrt(max(n, 1)) * (np.abs(v).max() if n else 1)


@pytest.mark.parametrize("scheme,D,group", [(O.Q_I8_SYM, 1024, 64), (O.Q_I8_ASYM, 272, 16), (O.Q_I4_SYM, 256, 32)])
def test_quant_scatter_routed(dev, scheme, D, group):
    """The same planes as quant_scatter leaves for the repeated K rows and the gathered V rows, dropped slots and
    caches outside the pool among them."""
    import torch
    from pikv_amd import ops
    r = rng(D)
    E, T, k = 3, 45, 2
    keys, vals = (to_dev(r.standard_normal(s).astype(np.float32), dev) for s in ((T, D), (E, T, D)))
    cid = r.integers(0, E, T * k).astype(np.int32)
    slot = np.array([np.count_nonzero(cid[:i] == c) for i, c in enumerate(cid)], dtype=np.int32)
    slot[::7] = -1
    pools = [ops.CachePool([20, 25, 9], 1, D, group, scheme, dev) for _ in range(2)]
    odd = cid.copy()
    odd[5], slot[5] = E + 4, 3
    idx, sl = to_dev(odd, dev), to_dev(slot, dev)
    pools[0].quant_scatter_routed(keys, vals, idx, sl, k, now=3.0)
    tok = torch.arange(T, device=dev).repeat_interleave(k)
    pools[1].quant_scatter(keys[tok].contiguous(), vals[to_dev(cid, dev).long(), tok].contiguous(), idx, sl, 1, now=3.0)
    for a, b in zip(pools[0].planes(), pools[1].planes()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,S,H,E,k,mask", [(1, 1, 128, 1, 1, False), (2, 33, 256, 4, 2, True), (3, 70, 384, 13, 8, False)])
def test_adaptive_router_native(dev, B, S, H, E, k, mask):
    """The native pass against the module's torch path (taken with autograd on): same selection, values to the
    rounding of float32 sums of H products."""
    import torch
    from pikv_amd.routing_strategy import AdaptiveRouter
    torch.manual_seed(H + E)
    m = AdaptiveRouter(H, E, top_k=k).to(dev).eval()
    x = torch.randn(B, S, H, device=dev)
    em = torch.randn(E, device=dev) if mask else None
    ref = m(x, em)
    with torch.no_grad():
        assert m._native(x, em)
        got = m(x, em)
        handle = m.load_balancing_router.router[0].register_forward_hook(lambda *a: None)
        assert not m._native(x, em)
        handle.remove()
        assert not m._native(x.double(), em) and not m._native(x[:, :, ::2], em)
    for a, b in zip(got, ref):
        assert a.shape == b.shape and a.dtype == b.dtype
    assert (got[1] == ref[1]).float().mean() > 0.99
    for i in (0, 3, 4):
        if E > 1 or i != 3:                              # one expert: the spread of one value, NaN on both sides
            assert torch.allclose(got[i], ref[i], rtol=0, atol=64 * 2.0 ** -24 * np.sqrt(H))
    same = (got[1] == ref[1]).all(-1)
    assert torch.allclose(got[2][same], ref[2][same], atol=64 * 2.0 ** -24 * np.sqrt(H))


@pytest.mark.parametrize("T,H,E,native", [(2048, 512, 64, True), (2049, 512, 64, False), (128, 2048, 8, True),
                                          (129, 2048, 8, False), (1, 2176, 2, False)])
def test_adaptive_router_size_rule(dev, T, H, E, native):
    """Both sides of the sizes where the native pass ends: one selection, values to the rounding of the sums."""
    import torch
    from pikv_amd.routing_strategy import AdaptiveRouter
    torch.manual_seed(T + H)
    m = AdaptiveRouter(H, E, top_k=2).to(dev).eval()
    x = torch.randn(1, T, H, device=dev)
    ref = m(x)
    with torch.no_grad():
        assert m._native(x, None) is native
        got = m(x)
    assert (got[1] == ref[1]).float().mean() > 0.99
    for i in (0, 3, 4):
        assert torch.allclose(got[i], ref[i], rtol=0, atol=64 * 2.0 ** -24 * np.sqrt(H))


@pytest.mark.parametrize("H,policy,seqs,seq", [(128, "lru", 2, 37), (256, "h2o", 2, 37), (640, "lru", 6, 70)])
def test_moe_native_forward_equals_module_path(dev, H, policy, seqs, seq):
    """PiKVMoE without autograd through the native experts and through the modules (a hook on one expert); 640 x 420 rows
    take the key projection from the library.  Logits to float32 sums; the cached rows are quantised from values that differ
    by a rounding, so a code may move by one: within a scale of each other, and nearly all equal."""
    import torch
    from pikv_amd import dense, moe
    from pikv_amd.config import config
    from pikv_amd.scheduling import SchedulingPolicy
    saved = dict(config)
    try:
        config.update(hidden_size=H, num_experts=3, kv_cache_size=60, kv_heads=2, kv_quant="int8", kv_group=128 if H == 640 else None,
                      vocab_size=512, cache_decrement=5, top_k=2, capacity_factor=1.5)
        assert dense.key_projection_pays(seqs * seq, H) is (H != 640)
        pol = SchedulingPolicy.H2O if policy == "h2o" else SchedulingPolicy.LRU
        models, native = [], [0, 0]
        for i in range(2):
            torch.manual_seed(1)
            m = moe.PiKVMoE(use_cache_scheduling=True, cache_scheduling_policy=pol).to(dev).eval()
            with torch.no_grad():
                for e in m.experts:
                    e.lora.lora_B.normal_(0.0, 0.05)
                for c in m.kv_caches:
                    c.value_lora.lora_B.normal_(0.0, 0.05)
                m.key_lora.lora_B.normal_(0.0, 0.05)

            def counted(*a, i=i, inner=m._experts_forward):
                native[i] += 1
                return inner(*a)
            m._experts_forward = counted
            models.append(m)
        models[1].experts[0].register_forward_hook(lambda *a: None)
        ids = torch.randint(512, (seqs, seq), device=dev)
        with torch.no_grad():
            for _ in range(3):
                a, b = (m(ids) for m in models)
                assert torch.allclose(a, b, rtol=0, atol=1e-5 * float(b.abs().max()))
        assert native == [3, 0]
        pa, pb = (m.pool for m in models)
        assert torch.equal(pa.fill, pb.fill) and int(pa.fill.min()) > 0
        live = torch.cat([base + torch.arange(int(n), device=dev) for base, n in zip(pa.base_host, pa.fill.tolist())])
        for which in ("k", "v"):
            ra, rb = (p.gather_dequant(which)[live] for p in (pa, pb))
            scale = getattr(pb, which + "_scale")[live].repeat_interleave(pb.group, dim=1)
            assert ((ra - rb).abs() <= 1.001 * scale).all()
            assert ((ra - rb).abs() > 0.5 * scale).float().mean() < 0.01
        assert torch.equal(pa.ts[live], pb.ts[live])
        assert torch.allclose(pa.acc[live], pb.acc[live], rtol=1e-3, atol=1e-5)
    finally:
        config.clear()
        config.update(saved)


@pytest.mark.parametrize("T,hidden,heads,kv,native", [(64, 1024, 32, 32, True), (65, 1024, 32, 32, False),
                                                      (32, 3584, 56, 14, True), (33, 3584, 56, 14, False), (1, 3712, 2, 2, False)])
def test_projection_size_rule(dev, monkeypatch, T, hidden, heads, kv, native):
    """Both sides of the sizes where the projections end to be one launch: the modules' values to float32 sums."""
    import torch
    from pikv_amd import ops
    from pikv_amd.attention import PiKVAttention
    torch.manual_seed(T + hidden)
    layer = PiKVAttention(hidden, heads, head_dim=64, num_kv_heads=kv, cache_size=8).to(dev).eval()
    calls, group = [], ops.linear_group
    monkeypatch.setattr(ops, "linear_group", lambda *a, **kw: calls.append(1) or group(*a, **kw))
    x = torch.randn(1, T, hidden, device=dev)
    with torch.no_grad():
        for got, m in zip(layer._project(x), (layer.q_proj, layer.k_proj, layer.v_proj)):
            want = m(x).view(got.shape)
            assert torch.allclose(got, want, rtol=0, atol=16 * 2.0 ** -24 * np.sqrt(hidden) * float(want.abs().max()))
    assert bool(calls) is native


@pytest.mark.parametrize("T,hidden,heads,kv,native", [
    (255, 1024, 32, 8, False), (256, 1024, 32, 8, True),
    (1112, 2048, 16, 4, True), (1113, 2048, 16, 4, False),       # 3.5e9 multiply-adds
    (330, 3072, 32, 8, False),                                   # ... of half empty rounds
    (871, 3072, 32, 16, False), (892, 3072, 32, 16, True), (1024, 3072, 32, 16, True), (1025, 3072, 32, 16, False)])   # one round
def test_tiled_projection_size_rule(dev, monkeypatch, T, hidden, heads, kv, native):
    """Both sides of the sizes where the projections of many tokens are one launch: the modules' values to float32 sums."""
    import torch
    from pikv_amd import ops
    from pikv_amd.attention import PiKVAttention
    torch.manual_seed(T + hidden)
    layer = PiKVAttention(hidden, heads, head_dim=64, num_kv_heads=kv, cache_size=8).to(dev).eval()
    calls, tiled = [], ops.linear_tiled
    monkeypatch.setattr(ops, "linear_tiled", lambda *a, **kw: calls.append(1) or tiled(*a, **kw))
    monkeypatch.setattr(ops, "linear_group", lambda *a, **kw: calls.append(2))
    x = torch.randn(1, T, hidden, device=dev)
    with torch.no_grad():
        for got, m in zip(layer._project(x), (layer.q_proj, layer.k_proj, layer.v_proj)):
            want = m(x).view(got.shape)
            assert torch.allclose(got, want, rtol=0, atol=16 * 2.0 ** -24 * np.sqrt(hidden) * float(want.abs().max()))
    assert calls == [1] * native


def test_native_prompt_attention_leaves_other_calls_alone(dev):
    """Hooks, dropout, masks, gradients, other types and forward-mode tangents keep the torch path; the two paths agree
    on what both take (float32 sums of some 200 products: 1e-5 of outputs of order one)."""
    import torch
    from torch.autograd import forward_ad
    from pikv_amd.attention import PiKVAttention
    torch.manual_seed(0)
    layer = PiKVAttention(128, 4, head_dim=64, cache_size=64, num_kv_heads=2).to(dev).eval()
    q, k, v = (torch.randn(2, 9, h, 64, device=dev) for h in (4, 2, 2))
    with torch.no_grad():
        assert layer._native_prefill(q, k, v, None)
        assert not layer._native_prefill(q, k, v, torch.ones(2, 9, device=dev))
        assert not layer._native_prefill(q.bfloat16(), k.bfloat16(), v.bfloat16(), None)
        with forward_ad.dual_level():
            assert not layer._native_prefill(forward_ad.make_dual(q, q), k, v, None)
        handle = layer.attn_dropout.register_forward_hook(lambda *a: None)
        x = torch.randn(2, 9, 128, device=dev)
        assert not layer._native_prefill(q, k, v, None)
        want = [layer(x)[0] for _ in range(2)]           # the second call attends to the first one's rows
        handle.remove()
        layer.reset_cache()
        for w in want:
            assert torch.allclose(layer(x)[0], w, rtol=0, atol=1e-5)
        layer.train()
        assert not layer._native_prefill(q, k, v, None)
    layer.eval()
    assert not layer._native_prefill(q.requires_grad_(), k, v, None)


@pytest.mark.parametrize("S,masked,dtype", [(5, False, "float32"), (5, True, "float32"), (1, False, "float32"),
                                            (5, False, "bfloat16")])
def test_context_of_another_batch_size_is_refused(dev, S, masked, dtype):
    """On every path of a layer, the native ones among them, and nothing of the context is lost; an empty one is replaced."""
    import torch
    from pikv_amd.attention import PiKVAttention
    dt = getattr(torch, dtype)
    layer = PiKVAttention(128, 2, head_dim=64, cache_size=32).to(dev, dt).eval()
    x = torch.randn(3, S, 128, device=dev, dtype=dt)
    mask = torch.ones(3, S, device=dev) if masked else None
    with torch.no_grad():
        layer(x[:2].expand(2, S, 128).contiguous())
        with pytest.raises(ValueError):
            layer(x, attention_mask=mask)
        assert layer.cache_ptr.tolist() == [S, S]
        layer.reset_cache()
        layer(x, attention_mask=mask)
    assert layer.cache_ptr.tolist() == [S] * 3
