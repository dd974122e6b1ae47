"""GPU parity of the launch shapes small calls take: few caches, short caches, few blocks."""
import numpy as np
import pytest

import pikv_oracle as O
from test_gpu_attend import _decode_reference
from test_gpu_read_evict import _fill_pool
from util import np_of, rng, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_caches,cap,heads,hq", [
    (3, 200, 8, 32),      # one tile per block
    (2, 321, 1, 4),       # one kv head: always four tiles per block
    (5, 300, 2, 8),       # two kv heads: two tiles per block
    (70, 1030, 4, 16),    # enough blocks for more tiles each
])
def test_scores_8bit_tiles_per_block(dev, n_caches, cap, heads, hq):
    """8-bit matrix-core scores of batches that take 1, 2 or 4 tiles per block, against float64 on the
    dequantised rows (the bar of the score tests: 1e-3 of the row's root-mean-square)."""
    r = rng(n_caches + cap)
    lens = [cap - (37 * c) % (cap - 1) for c in range(n_caches)]
    pool, ref = _fill_pool(dev, r, [cap] * n_caches, lens, heads, 128, 128, O.Q_I8_SYM)
    q = O.bf16_round(r.standard_normal((n_caches, hq, 128)).astype(np.float32))
    scores, tmax, tsum = (np_of(t) for t in pool.scores(to_dev(q, dev, "bf16"), hq))
    for c in sorted({0, 1, n_caches // 2, n_caches - 1}):
        rows = ref.valid_rows(c)[:lens[c]]
        k_hat = O.dequantize_groups(ref.k_codes[rows], ref.k_scale[rows], ref.k_zero[rows], 128)
        want = O.attention_scores(q[c], k_hat, heads, 1.0 / np.sqrt(128))
        got = scores[c][:, :lens[c]]
        rms = np.sqrt((want.astype(np.float64) ** 2).mean())
        assert np.abs(got - want).max() <= 1e-3 * rms
        for t in range((lens[c] + 63) // 64):
            s = got[:, 64 * t:min(64 * t + 64, lens[c])].astype(np.float64)
            np.testing.assert_allclose(tmax[c, t], s.max(axis=1), rtol=1e-6)
            np.testing.assert_allclose(tsum[c, t], np.exp(s - s.max(axis=1, keepdims=True)).sum(axis=1), rtol=1e-4)


@pytest.mark.parametrize("scheme,qdtype", [(O.Q_I8_SYM, "bf16"), (O.Q_I4_ASYM, "bf16"), (O.Q_I4_SYM, "f32")])
@pytest.mark.parametrize("length", [1, 63, 65, 129, 1985, 2049, 4161])
def test_decode_attend_few_ranges(dev, scheme, qdtype, length):
    """One and two caches on their own: ranges of one or two tiles, 1 to 66 of them per cache - the merge with
    one wavefront per head and, from 32 ranges on, with four.  Bars of test_decode_attend_one_call."""
    heads, hq, group = 4, 16, (128 if scheme == O.Q_I8_SYM else 32)
    r = rng(length)
    lens = [length, max(1, length // 3)]
    pool, ref = _fill_pool(dev, r, [length + 3] * 2, lens, heads, 128, group, scheme)
    acc0 = r.random(pool.rows).astype(np.float32)
    pool.acc.copy_(to_dev(acc0, dev))
    q = r.standard_normal((2, hq, 128)).astype(np.float32) * 2
    q = O.bf16_round(q) if qdtype == "bf16" else q
    out = np_of(pool.decode_attend(to_dev(q, dev, qdtype), hq, now=4.0))
    want, acc = _decode_reference(ref, q, lens, acc0, heads, group, 1.0 / np.sqrt(128), 1.0)
    for c in range(2):
        rms = np.sqrt((want[c].astype(np.float64) ** 2).mean()) + 1e-12
        assert np.abs(out[c] - want[c]).max() <= 1e-3 * rms
    np.testing.assert_allclose(np_of(pool.acc), acc, rtol=1e-3, atol=1e-5)


@pytest.mark.parametrize("policy", ["h2o", "h2o_leave_room", "lru", "all"])
@pytest.mark.parametrize("caps,D,heavy,recent", [
    ([128, 118, 1, 90], 64, 0.1, 0.1),          # selected and compacted by one block per cache
    ([1024, 1500, 1025], 2048, 0.5, 0.3),       # selected by one block, more than a megabyte of survivors
    ([1024, 1500, 1025], 2048, -0.5, 0.8),      # a ratio below zero: one row of that set
    ([200, 190, 170], 2048, 0.9, 0.05),         # wide rows: between two thirds of a megabyte and one
    ([150, 140, 100], 2048, 0.9, 0.05),         # ... and below
    ([8192, 8000], 32, 0.06, 0.01),             # the longest caches of the one-block form
    ([9000, 5000], 32, 0.1, 0.05),              # several blocks per cache
])
def test_make_room_and_append(dev, policy, caps, D, heavy, recent):
    """make_room(append=True) + append_rows: survivors of every overflowing cache and their order against the
    restatement's selections, exact; caches with the space keep every row; then the new rows behind them."""
    import torch
    from pikv_amd import ops
    r = rng(len(caps) + D)
    n_add = 7
    fills = [max(1, c - (3 if i % 2 == 0 else 40)) for i, c in enumerate(caps)]   # every other cache overflows
    pool = ops.CachePool(caps, 1, D, min(D, 1024), ops.Q_I8_SYM, dev)
    pool.k_codes.random_(-127, 127), pool.v_codes.random_(-127, 127)
    acc = np.round(r.random(pool.rows) * 50).astype(np.float32)                   # many ties
    ts = r.permutation(pool.rows).astype(np.float32)
    pool.acc.copy_(to_dev(acc, dev)), pool.ts.copy_(to_dev(ts, dev))
    pool.fill.copy_(to_dev(np.array(fills, np.int32), dev))
    before_k, before_v = np_of(pool.k_codes), np_of(pool.v_codes)
    code = {"lru": ops.EVICT_LRU, "all": ops.EVICT_ALL}.get(policy, ops.EVICT_H2O)
    pool.make_room(code, count_all=n_add, heavy_ratio=heavy, recent_ratio=recent, leave_room=policy == "h2o_leave_room",
                   append=True)
    kn, vn = r.standard_normal((len(caps) * n_add, D)).astype(np.float32), r.standard_normal((len(caps) * n_add, D)).astype(np.float32)
    pool.append_rows(to_dev(kn, dev), to_dev(vn, dev), now=9.0)
    k, v, acc2, ts2 = (np_of(t) for t in (pool.k_codes, pool.v_codes, pool.acc, pool.ts))
    new_codes = O.quantize_groups(kn, min(D, 1024), O.Q_I8_SYM)[0]
    for c, (cap, L) in enumerate(zip(caps, fills)):
        base, n = int(pool.row_base[c]), min(n_add, cap)
        over = L + n - cap
        a, t = acc[base:base + L], ts[base:base + L]
        keep = np.ones(L, bool)
        if over > 0 and policy == "lru":
            keep = O.lru_keep(t, min(over, L))
        elif over > 0 and policy == "all":
            keep[:] = False
        elif over > 0:
            nh, nr = O.h2o_budget(L, heavy, recent)
            if policy == "h2o_leave_room":
                nh = min(nh, cap - n)
                nr = min(nr, cap - n - nh)
            keep = O.h2o_keep(a, t, nh, nr)
        rows = base + np.nonzero(keep)[0]
        m = len(rows)
        assert int(pool.new_len[c]) == m and int(pool.fill[c]) == min(m + n, cap), c
        assert np.array_equal(k[base:base + m], before_k[rows]) and np.array_equal(v[base:base + m], before_v[rows]), c
        assert np.array_equal(acc2[base:base + m], acc[rows]) and np.array_equal(ts2[base:base + m], ts[rows]), c
        w = min(n_add, cap - m)
        assert np.array_equal(k[base + m:base + m + w].astype(np.int16), new_codes[c * n_add:c * n_add + w]), c
        assert (ts2[base + m:base + m + w] == 9.0).all() and (acc2[base + m:base + m + w] == 0.0).all()


@pytest.mark.parametrize("caps,rows", [([9, 40, 3, 64], 1), ([9, 40, 3, 64], 5), ([300] * 3, 299), ([0, 7], 7)])
@pytest.mark.parametrize("D,scheme", [(64, O.Q_I8_SYM), (96, O.Q_I4_ASYM), (2048, O.Q_I8_ASYM)])
def test_append_rows_advances_with_the_write(dev, caps, rows, D, scheme):
    """append_rows(advance=True) behind a plain make_room leaves what make_room(append=True) + append_rows does; a
    write that is refused leaves the fill at the rows that are there."""
    import torch
    from pikv_amd import ops
    r = rng(D + rows)
    pools = [ops.CachePool(caps, 1, D, 32, scheme, dev) for _ in range(2)]
    fills = np.array([max(0, c - 3) for c in caps], np.int32)
    k, v = (to_dev(r.standard_normal((len(caps) * rows, D)).astype(np.float32), dev) for _ in range(2))
    for pool, append in zip(pools, (True, False)):
        pool.fill.copy_(to_dev(fills, dev))
        pool.make_room(ops.EVICT_LRU, count_all=rows, append=append)
    held = pools[1].fill.clone()
    assert torch.equal(held, pools[1].new_len)
    with pytest.raises(ValueError):
        pools[1].append_rows(k, v[:-1], now=2.0, advance=True)
    assert torch.equal(pools[1].fill, held)
    pools[0].append_rows(k, v, now=2.0)
    pools[1].append_rows(k, v, now=2.0, advance=True)
    for a, b in zip([pools[0].fill, *pools[0].planes()], [pools[1].fill, *pools[1].planes()]):
        assert torch.equal(a, b)


def test_attention_cache_after_a_refused_write(dev):
    """A layer whose new rows are refused claims none of them."""
    import torch
    from pikv_amd.attention import PiKVAttention
    layer = PiKVAttention(128, 2, head_dim=64, cache_size=16).to(dev).eval()
    x = torch.randn(2, 5, 128, device=dev)
    with torch.no_grad():
        layer(x)
        k = torch.randn(2, 4, 2, 64, device=dev)
        with pytest.raises(ValueError):
            layer._update_cache(k, k[:, :3])
        assert layer.cache_ptr.tolist() == [5, 5]
        layer._update_cache(k, k)
    assert layer.cache_ptr.tolist() == [9, 9]


@pytest.mark.parametrize("scheme,heads,hq,dh,group", [
    (O.Q_I8_SYM, 2, 4, 128, 128), (O.Q_I8_ASYM, 4, 4, 64, 32), (O.Q_I4_ASYM, 2, 6, 64, 32), (O.Q_I4_SYM, 1, 7, 128, 64)])
@pytest.mark.parametrize("S,lens", [(1, [5]), (2, [0, 33]), (31, [1, 64]), (33, None), (70, [32, 300]), (5, [1500])])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_attend(dev, scheme, heads, hq, dh, group, S, lens, causal):
    """Chunks around the 32-row and 32-key tiles, over no cached rows, a few, and enough for several blocks a row,
    against float64.  Bound: a score is a float32 sum of d products, off by some 2^-24 sqrt(d) of the largest score
    (the cached rows have channels 20 times the others), which is the relative error of its probability; the output
    averages n values by them.  4 * 2^-24 * sqrt(d + n) * (1 + largest score) of the largest value covers both."""
    from pikv_amd import ops
    r = rng(S * 131 + dh + hq)
    B = 2 if lens is None else len(lens)
    D = heads * dh
    q, k, v = (r.standard_normal((B, S, h, dh)).astype(np.float32) for h in (hq, heads, heads))
    pool = ref = None
    if lens is not None:
        pool, ref = _fill_pool(dev, r, [max(lens) + 3] * B, lens, heads, dh, group, scheme)
    got = np_of(ops.prefill_attend(*(to_dev(t, dev, "f32") for t in (q, k, v)), pool, causal)).astype(np.float64)
    for b in range(B):
        n = 0 if lens is None else lens[b]
        kk, vv = k[b].astype(np.float64), v[b].astype(np.float64)
        if n:
            rows = ref.valid_rows(b)[:n]
            past = [O.dequantize_groups(c[rows], s[rows], z[rows], group).reshape(n, heads, dh)
                    for c, s, z in ((ref.k_codes, ref.k_scale, ref.k_zero), (ref.v_codes, ref.v_scale, ref.v_zero))]
            kk, vv = np.concatenate([past[0], kk]), np.concatenate([past[1], vv])
        for h in range(hq):
            s = q[b, :, h].astype(np.float64) @ kk[:, h // (hq // heads)].T / np.sqrt(dh)
            size = (1.0 + np.abs(s).max()) * np.abs(vv).max()
            if causal:
                s[np.arange(n + S)[None, :] > n + np.arange(S)[:, None]] = -np.inf
            p = np.exp(s - s.max(axis=1, keepdims=True))
            want = (p / p.sum(axis=1, keepdims=True)) @ vv[:, h // (hq // heads)]
            assert np.abs(got[b, :, h] - want).max() <= 4 * 2.0 ** -24 * np.sqrt(dh + n + S) * size


@pytest.mark.parametrize("dh,scheme", [(64, O.Q_I4_SYM), (128, O.Q_I8_SYM)])
def test_prefill_attend_takes_views(dev, dh, scheme):
    """Rows that begin one, two and three floats into a buffer give what the same rows give in a buffer of their own."""
    import torch
    from pikv_amd import ops
    r = rng(dh)
    q, k, v = (to_dev(r.standard_normal((2, 37, h, dh)).astype(np.float32), dev) for h in (4, 2, 2))
    pool, _ = _fill_pool(dev, r, [40] * 2, [40, 7], 2, dh, 32, scheme)
    want = ops.prefill_attend(q, k, v, pool)
    views = []
    for i, t in enumerate((q, k, v)):
        buf = torch.empty(t.numel() + 4, device=dev)
        views.append(buf[i + 1:i + 1 + t.numel()].view(t.shape).copy_(t))
        assert views[-1].data_ptr() % 16
    assert torch.equal(ops.prefill_attend(*views, pool), want)


@pytest.mark.parametrize("dh", [64, 128])
def test_prefill_attend_nan_rows_and_unaligned_output(dev, dh):
    """A NaN or infinite query makes its own output NaN and no other; an output that begins between 16 bytes holds the same
    values, and nothing beside it is written."""
    import torch
    from pikv_amd import _native as N, ops
    r = rng(dh + 1)
    q, k, v = (to_dev(r.standard_normal((2, 45, h, dh)).astype(np.float32), dev) for h in (4, 2, 2))
    pool, _ = _fill_pool(dev, r, [70] * 2, [70, 9], 2, dh, 32, O.Q_I4_ASYM)
    want = ops.prefill_attend(q, k, v, pool)
    bad = q.clone()
    bad[0, 7, 1, 3], bad[1, 44, 2, 0] = float("nan"), float("inf")
    got = ops.prefill_attend(bad, k, v, pool)
    hit = torch.zeros(2, 45, 4, 1, dtype=torch.bool, device=dev)
    hit[0, 7, 1], hit[1, 44, 2] = True, True
    assert bool(got.isnan().eq(hit).all()) and torch.equal(torch.where(hit, want, got), want)
    buf = torch.full((q.numel() + 2,), 7.0, device=dev)
    p = lambda t: t.data_ptr()
    N.call("pikv_prefill_attend", p(q), p(k), p(v), 2, 45, 2, 4, dh, 1, dh ** -0.5, *map(p, (*pool._planes("k"), *pool._planes("v"))),
           pool.scheme, pool.group, p(pool.row_base), p(pool.fill), pool.max_cap, p(buf) + 4, None, 0,
           torch.cuda.current_stream().cuda_stream)
    assert torch.equal(buf[1:-1].view_as(want), want) and float(buf[0]) == float(buf[-1]) == 7.0


@pytest.mark.parametrize("A", [1, 255, 512, 513, 4095, 4096, 4097, 8191, 8192, 8193, 16000])
@pytest.mark.parametrize("E,capacity", [(1, 5000), (8, 700), (64, 90)])
def test_capacity_slots_chunks(dev, A, E, capacity):
    """Slots and totals on both sides of the lengths where blocks count the assignments before them by themselves,
    ids out of range among them."""
    from pikv_amd import ops
    r = rng(A + E)
    idx = r.integers(0, E, A).astype(np.int32)
    idx[3::97] = E
    idx[5::89] = -1
    slot, count = (np_of(t) for t in ops.capacity_slots(to_dev(idx, dev), E, capacity))
    seen = np.zeros(E, dtype=np.int64)
    for a, e in enumerate(idx):
        want = -1
        if 0 <= e < E:
            want = seen[e] if seen[e] < capacity else -1
            seen[e] += 1
        assert slot[a] == want
    assert np.array_equal(count, seen)


@pytest.mark.parametrize("cap,lens,hq", [(64, [64, 0], 1), (2048, [2048, 65], 64), (2049, [2049, 1], 64),
                                         (2048, [1983, 64], 65)])
@pytest.mark.parametrize("write_probs", [False, True])
def test_h2o_accumulate_own_statistics(dev, cap, lens, hq, write_probs):
    """On both sides of 32 tiles and 64 heads, where the accumulation merges the tile statistics by itself: importance,
    accumulators, probabilities and head statistics against float64.  Probabilities are float32 exponentials of score
    differences below 30: 2^-24 * 30 of each, with a factor of four."""
    from pikv_amd import ops
    import torch
    r = rng(cap + hq)
    pool = ops.CachePool([cap] * 2, 1, 64, 64, O.Q_I8_SYM, dev)
    pool.fill.copy_(torch.tensor(lens, dtype=torch.int32))
    s = (4 * r.standard_normal((2, hq, cap))).astype(np.float32)
    n_tiles = (cap + 63) // 64
    tmax = np.full((2, n_tiles, hq), -np.inf, dtype=np.float32)
    tsum = np.zeros((2, n_tiles, hq), dtype=np.float32)
    for c, n in enumerate(lens):
        for t in range((n + 63) // 64):
            x = s[c, :, 64 * t:min(64 * t + 64, n)].astype(np.float64)
            tmax[c, t] = x.max(axis=1)
            tsum[c, t] = np.exp(x - x.max(axis=1, keepdims=True)).sum(axis=1)
    sd = to_dev(s, dev)
    imp = np_of(pool.h2o_accumulate(sd, to_dev(tmax, dev), to_dev(tsum, dev), now=2.0, write_probs=write_probs,
                                    return_importance=True))
    stats, acc, ts, probs = np_of(pool.head_stats), np_of(pool.acc), np_of(pool.ts), np_of(sd)
    tol = 4 * 30 * 2.0 ** -24
    for c, n in enumerate(lens):
        if n == 0:
            assert not acc[c * cap:(c + 1) * cap].any() and np.isneginf(stats[c, :, 0]).all()
            continue
        x = s[c, :, :n].astype(np.float64)
        p = np.exp(x - x.max(axis=1, keepdims=True))
        np.testing.assert_allclose(stats[c, :, 0], x.max(axis=1), rtol=0)
        np.testing.assert_allclose(stats[c, :, 1], p.sum(axis=1), rtol=tol)
        p /= p.sum(axis=1, keepdims=True)
        np.testing.assert_allclose(imp[c, :n], p.sum(axis=0), rtol=tol)
        np.testing.assert_allclose(acc[c * cap:c * cap + n], p.sum(axis=0), rtol=tol)
        assert (ts[c * cap:c * cap + n] == 2.0).all() and not acc[c * cap + n:(c + 1) * cap].any()
        if write_probs:
            np.testing.assert_allclose(probs[c, :, :n], p, rtol=tol)
