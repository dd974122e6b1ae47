"""The work a user of pikv_amd has it do, as timed cases: each goes through the public entry points the way a
serving or training program calls them.

Kinds of cases (the "kind" of a case; the other fields are its sizes and options):

  prefill    one prompt batch: fused router -> quantise + scatter into the routed caches -> advance -> scores of
             one query per cache -> H2O importance (the step of bench.py)
  route      mixture-of-experts routing of a long token stream: fused router with bias and per-expert logit
             scale -> quantise + scatter into caches sized by the observed load
  decode     one decode step of a batch of sequences: append a token each -> one-call decode read with the H2O
             bookkeeping
  attention  PiKVAttention as a layer of a model: a prompt in one or more chunks, or a single new token over a
             cached context
  moe        PiKVMoE on token ids: inference, or a training step with the gradients of every parameter
  evict      H2O or LRU eviction of a batch of caches: selection + in-place compaction
  pyramid    long-context compression: per-layer top-k of the tokens by score, then quantisation

Sizes come from bench.py, the tests and config.py.  listed() names the ones that stand for a use; draw() spreads
over the same ranges.
"""
import math

import torch

from pikv_amd import attention, moe, ops, pyramid
from pikv_amd.config import config
from pikv_amd.scheduling import SchedulingPolicy

SCHEMES = {"int8": ops.Q_I8_SYM, "int8_asym": ops.Q_I8_ASYM, "int4": ops.Q_I4_ASYM, "int4_sym": ops.Q_I4_SYM}
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}

# (kv heads, query heads, head_dim) of the cache geometries bench.py reads
GEOMETRIES = [(8, 32, 128), (8, 64, 128), (32, 32, 128), (40, 40, 128), (4, 28, 128), (2, 16, 128), (2, 12, 128),
              (2, 14, 64), (8, 40, 128), (2, 32, 128), (12, 12, 64), (16, 16, 64), (25, 25, 64), (8, 32, 64),
              (8, 24, 128), (16, 16, 256), (8, 16, 256), (1, 71, 64), (4, 36, 128), (1, 48, 128)]


def listed():
    return [
        # the small single-device configuration, a forward over token ids: all launches, hardly any bytes
        dict(name="moe_small", kind="moe", batch=2, seq=64, hidden=256, experts=4, slots=128, policy="lru",
             quant="int8", train=False),
        # a training step of the same model at a batch in between: forward, loss, backward
        dict(name="moe_train", kind="moe", batch=8, seq=96, hidden=256, experts=4, slots=512, policy="h2o",
             quant="int8", train=True),
        # a short ragged prompt batch on a GQA model, the caches per head and token in 8 bits
        dict(name="prefill_short", kind="prefill", batch=3, seq=577, hidden=2048, experts=8, top_k=2,
             kv_heads=8, q_heads=32, head_dim=128, slots=1024, quant="int8", group=128, dtype="bf16"),
        # the prefill compress-write workload of bench.py: 32768 tokens, 32 heads x 128
        dict(name="prefill_long", kind="prefill", batch=16, seq=2048, hidden=4096, experts=8, top_k=2,
             kv_heads=32, q_heads=32, head_dim=128, slots=8192, quant="int8", group=128, dtype="bf16"),
        # wide routing: 64 experts, top 8, popularity after Zipf
        dict(name="route_wide", kind="route", tokens=65536, hidden=7168, experts=64, top_k=8, kv_heads=8,
             head_dim=128, quant="int8", group=128, dtype="bf16"),
        # one user, a short context: what a decode step costs when it is all latency
        dict(name="decode_single", kind="decode", batch=1, context=700, ragged=0.0, kv_heads=8, q_heads=32,
             head_dim=128, quant="int4", group=32, dtype="bf16"),
        # an ordinary serving batch: sequences of all lengths up to some thousands, 8-bit caches, 7 heads per kv head
        dict(name="decode_ragged", kind="decode", batch=24, context=4000, ragged=0.9, kv_heads=4, q_heads=28,
             head_dim=128, quant="int8", group=128, dtype="bf16"),
        # the decode read of bench.py: 64 sequences x 32768 tokens, 4-bit in groups of 32
        dict(name="decode_long", kind="decode", batch=64, context=32768, ragged=0.0, kv_heads=8, q_heads=32,
             head_dim=128, quant="int4", group=32, dtype="bf16"),
        # the attention module in float32 (the dtype it is created in): a new token over a cached context
        dict(name="attention_token", kind="attention", batch=8, chunk=1, chunks=1, context=3000, hidden=1024,
             kv_heads=16, q_heads=16, head_dim=64, quant="int4", group=32),
        # the same module over a prompt that comes in two chunks, the second attends to the first as it was cached
        dict(name="attention_prompt", kind="attention", batch=2, chunk=500, chunks=2, context=0, hidden=2048,
             kv_heads=8, q_heads=16, head_dim=128, quant="int8", group=128),
        # caches of the decode read down to 1/16 heavy and 1/128 recent rows
        dict(name="evict_h2o", kind="evict", policy="h2o", batch=64, context=32768, kv_heads=8, head_dim=128,
             quant="int4", group=32),
        # pyramid compression of a long context: 32 layers, budget from 100 % down to 25 %
        dict(name="pyramid", kind="pyramid", layers=32, tokens=131072, kv_heads=8, head_dim=128, quant="int8",
             group=128, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _quant(rng, head_dim):
    q = rng.choice(["int8", "int8", "int8_asym", "int4", "int4", "int4_sym"])
    return q, (32 if q.startswith("int4") else head_dim)


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "route", "decode", "decode", "decode", "attention", "attention", "moe",
                       "moe", "evict", "pyramid"])
    if kind == "prefill":
        dh = rng.choice([64, 128])
        quant, group = _quant(rng, dh)
        kv = rng.choice([4, 8, 16, 32])
        batch, seq = rng.randint(1, 16), _log_int(rng, 40, 2048)
        experts = rng.choice([4, 8, 16])
        return dict(kind=kind, batch=batch, seq=seq, hidden=256 * rng.randint(1, 16), experts=experts, top_k=2,
                    kv_heads=kv, q_heads=kv * rng.choice([1, 1, 4]), head_dim=dh,
                    slots=max(64, int(batch * seq * 2.4 / experts)), quant=quant, group=group,
                    dtype=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "route":
        quant, group = _quant(rng, 128)
        return dict(kind=kind, tokens=_log_int(rng, 500, 65536), hidden=512 * rng.randint(2, 14),
                    experts=rng.choice([16, 32, 64]), top_k=rng.randint(2, 8), kv_heads=rng.choice([2, 4, 8]),
                    head_dim=128, quant=quant, group=group, dtype=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "decode":
        kv, hq, dh = rng.choice(GEOMETRIES)
        quant, group = _quant(rng, dh)
        batch, context = _log_int(rng, 1, 64), _log_int(rng, 200, 32768)
        while batch * context * kv * dh > (64 * 8192 * 8 * 128):   # a quarter of the largest read
            context = max(200, context // 2)
        return dict(kind=kind, batch=batch, context=context, ragged=rng.choice([0.0, 0.5, 0.9]), kv_heads=kv,
                    q_heads=hq, head_dim=dh, quant=quant, group=group, dtype=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "attention":
        kv, hq, dh = rng.choice([(4, 8, 128), (8, 16, 128), (12, 12, 64), (16, 16, 64), (8, 32, 64), (8, 32, 128)])
        quant, group = _quant(rng, dh)
        one = rng.random() < 0.5
        return dict(kind=kind, batch=rng.randint(1, 16 if one else 4), chunk=1 if one else _log_int(rng, 33, 1000),
                    chunks=1 if one else rng.randint(1, 2), context=_log_int(rng, 200, 6000) if one else 0,
                    hidden=256 * rng.randint(2, 12), kv_heads=kv, q_heads=hq, head_dim=dh, quant=quant, group=group)
    if kind == "moe":
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_log_int(rng, 16, 256), hidden=128 * rng.choice([2, 4]),
                    experts=rng.choice([4, 6]), slots=_log_int(rng, 100, 1000), policy=rng.choice(["lru", "h2o"]),
                    quant=rng.choice(["int8", "int8_asym"]), train=rng.random() < 0.5)
    if kind == "evict":
        quant, group = _quant(rng, 128)
        batch, context = _log_int(rng, 1, 64), _log_int(rng, 300, 32768)
        return dict(kind=kind, policy=rng.choice(["h2o", "h2o", "lru"]), batch=batch, context=context,
                    kv_heads=rng.choice([2, 4, 8]), head_dim=128, quant=quant, group=group)
    quant, group = _quant(rng, 128)
    return dict(kind=kind, layers=rng.randint(4, 32), tokens=_log_int(rng, 4000, 60000), kv_heads=rng.choice([2, 4, 8]),
                head_dim=128, quant=quant, group=group, dtype=rng.choice(["bf16", "bf16", "f32"]))


# ---- inputs ---------------------------------------------------------------------------------------------------

def _dev():
    return torch.device("cuda:0")


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device=_dev()).to(dtype)


def _kv_rows(g, n, D, dtype):
    """K or V rows: normal, one channel in a hundred twenty times as large."""
    t = torch.randn(n, D, generator=g, device=_dev())
    ch = torch.randperm(D, generator=g, device=_dev())[:max(1, D // 100)]
    t[:, ch] *= 20.0
    return t.to(dtype)


def _lengths(c):
    """Rows of every sequence: the longest is `context`, the others spread down to (1 - ragged) of it."""
    return [max(1, int(c["context"] * (1.0 - c["ragged"] * ((i * 0.618034) % 1.0)))) for i in range(c["batch"])]


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=_dev())


def _capacity(c):
    return int(c["batch"] * c["seq"] * 1.25 * c["top_k"] / c["experts"])


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _prepare_prefill(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    T, D = c["batch"] * c["seq"], c["kv_heads"] * c["head_dim"]
    pool = ops.CachePool([c["slots"]] * c["experts"], c["kv_heads"], c["head_dim"], c["group"], SCHEMES[c["quant"]], _dev())
    return dict(case=c, x=_randn(g, T, c["hidden"], dtype=dt), w=(0.02 * _randn(g, c["experts"], c["hidden"])).to(dt),
                k=_kv_rows(g, T, D, dt), v=_kv_rows(g, T, D, dt),
                q=_randn(g, c["experts"], c["q_heads"], c["head_dim"], dtype=dt), pool=pool, now=0.0)


def _run_prefill(s):
    c, pool = s["case"], s["pool"]
    cap = _capacity(c)
    s["now"] += 1.0
    pool.fill.zero_()
    r = ops.router_fused(s["x"], s["w"], top_k=c["top_k"], capacity=cap)
    pool.quant_scatter(s["k"], s["v"], r.topk_idx, r.slot, c["top_k"], now=s["now"])
    pool.advance(r.count, cap)
    scores, tile_max, tile_sum = pool.scores(s["q"], c["q_heads"])
    pool.h2o_accumulate(scores, tile_max, tile_sum, now=s["now"])
    return [r.probs, r.topk_idx, r.topk_w, r.slot, r.count, pool.fill, *pool.planes()]


def _expert_load(c, dt):
    """Popularity of the experts (Zipf, as a bias of the gate) and cache sizes with a quarter of headroom over the
    load that earlier tokens of another model have shown."""
    g, E, n = _gen(3), c["experts"], min(c["tokens"], 8192)
    pop = (torch.randperm(E, generator=g, device=_dev()).float() + 1) ** -1.2
    bias = (pop / pop.sum()).log()
    x, w = _randn(g, n, c["hidden"], dtype=dt), (0.02 * _randn(g, E, c["hidden"])).to(dt)
    count = ops.router_fused(x, w, bias, top_k=c["top_k"], capacity=n).count.float()
    scale = (1.0 / (count / count.mean()).clamp_min(0.1)).clamp(0.5, 2.0)
    count = ops.router_fused(x, w, bias, top_k=c["top_k"], capacity=n, expert_scale=scale).count
    return bias, [min(c["tokens"], int(1.25 * m * c["tokens"] / n) + 64) for m in count.tolist()]


def _prepare_route(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    T, E, D = c["tokens"], c["experts"], c["kv_heads"] * c["head_dim"]
    x, w = _randn(g, T, c["hidden"], dtype=dt), (0.02 * _randn(g, E, c["hidden"])).to(dt)
    bias, caps = _expert_load(c, dt)
    count = ops.router_fused(x, w, bias, top_k=c["top_k"], capacity=T).count.float()
    scale = (1.0 / (count / count.mean()).clamp_min(0.1)).clamp(0.5, 2.0)
    pool = ops.CachePool(caps, c["kv_heads"], c["head_dim"], c["group"], SCHEMES[c["quant"]], _dev())
    return dict(case=c, x=x, w=w, bias=bias, scale=scale, k=_randn(g, T, D, dtype=dt), v=_randn(g, T, D, dtype=dt),
                pool=pool, now=0.0)


def _run_route(s):
    c, pool = s["case"], s["pool"]
    s["now"] += 1.0
    pool.fill.zero_()
    r = ops.router_fused(s["x"], s["w"], s["bias"], top_k=c["top_k"], capacity=c["tokens"], expert_scale=s["scale"])
    pool.quant_scatter(s["k"], s["v"], r.topk_idx, r.slot, c["top_k"], now=s["now"])
    pool.advance(r.count)
    return [r.probs, r.topk_idx, r.topk_w, r.slot, r.count, pool.fill, *pool.planes()]


def _fill_pool(pool, lengths, g):
    """Normal K and V rows into the caches, some sequences at a time."""
    c = 0
    while c < len(lengths):
        some, rows = [], 0
        while c < len(lengths) and (not some or rows + lengths[c] <= 131072):
            some.append(c)
            rows += lengths[c]
            c += 1
        cid = torch.repeat_interleave(_i32(some), _i32([lengths[i] for i in some]))
        slot = torch.cat([torch.arange(lengths[i], dtype=torch.int32, device=_dev()) for i in some])
        pool.quant_scatter(_randn(g, rows, pool.D, dtype=torch.bfloat16), _randn(g, rows, pool.D, dtype=torch.bfloat16),
                           cid, slot, 1)
    pool.fill.copy_(_i32(lengths))


def _prepare_decode(c, seed):
    g, dt, B = _gen(seed), DTYPES[c["dtype"]], c["batch"]
    lens = [n - 1 for n in _lengths(c)]                 # this step's token comes on top
    pool = ops.CachePool([c["context"]] * B, c["kv_heads"], c["head_dim"], c["group"], SCHEMES[c["quant"]], _dev())
    _fill_pool(pool, lens, g)
    return dict(case=c, pool=pool, lens=_i32(lens), one=torch.ones(B, dtype=torch.int32, device=_dev()),
                seq=torch.arange(B, dtype=torch.int32, device=_dev()), slot=torch.zeros(B, dtype=torch.int32, device=_dev()),
                q=_randn(g, B, c["q_heads"], c["head_dim"], dtype=dt), k=_randn(g, B, pool.D, dtype=dt),
                v=_randn(g, B, pool.D, dtype=dt), now=0.0)


def _run_decode(s):
    c, pool = s["case"], s["pool"]
    s["now"] += 1.0
    pool.fill.copy_(s["lens"])                          # the batch of this step, as the server hands it over
    pool.quant_scatter(s["k"], s["v"], s["seq"], s["slot"], 1, now=s["now"])
    pool.advance(s["one"])
    out = pool.decode_attend(s["q"], c["q_heads"], now=s["now"])
    return [out, pool.fill, *pool.planes()]


def _prepare_attention(c, seed):
    g = _gen(seed)
    torch.manual_seed(int(seed))
    layer = attention.PiKVAttention(c["hidden"], c["q_heads"], head_dim=c["head_dim"],
                                    cache_size=c["context"] + c["chunk"] * c["chunks"] + 8, num_kv_heads=c["kv_heads"],
                                    kv_quant=c["quant"], kv_group=c["group"]).to(_dev()).eval()
    x = [_randn(g, c["batch"], c["chunk"], c["hidden"]) for _ in range(c["chunks"])]
    lens = None
    if c["context"]:
        past = [_randn(g, c["batch"], c["kv_heads"], c["context"], c["head_dim"]) for _ in range(2)]
        with torch.no_grad():
            layer.load_past_key_values(tuple(past), layout="hf")
        lens = layer.pool.fill.clone()
    return dict(case=c, layer=layer, x=x, lens=lens)


def _run_attention(s):
    layer = s["layer"]
    with torch.no_grad():
        if s["lens"] is not None:
            layer.pool.fill.copy_(s["lens"])            # back to the accepted tokens, then the next one
        else:
            layer.reset_cache()                         # a new prompt
        out = [layer(x)[0] for x in s["x"]]
    return [*out, layer.pool.fill, *layer.pool.planes()]


def _prepare_moe(c, seed):
    g = _gen(seed)
    config.update(hidden_size=c["hidden"], num_experts=c["experts"], kv_cache_size=c["slots"], kv_heads=4,
                  kv_quant=c["quant"], kv_group=None, vocab_size=50257, cache_decrement=10, top_k=2, capacity_factor=1.5)
    torch.manual_seed(int(seed))
    policy = SchedulingPolicy.H2O if c["policy"] == "h2o" else SchedulingPolicy.LRU
    model = moe.PiKVMoE(use_cache_scheduling=True, cache_scheduling_policy=policy).to(_dev())
    with torch.no_grad():
        for e in model.experts:
            e.lora.lora_B.normal_(0.0, 0.05)
    model.train(c["train"])
    ids = [torch.randint(50257, (c["batch"], c["seq"]), generator=g, device=_dev()) for _ in range(2)]
    state = dict(case=c, model=model, ids=ids[0], targets=ids[1])
    with torch.no_grad():
        model(ids[0])                                   # the caches of a program in use are not empty
    return state


def _run_moe(s):
    c, model = s["case"], s["model"]
    if not c["train"]:
        with torch.no_grad():
            logits = model(s["ids"])
        return [logits, model.pool.fill, *model.pool.planes()]
    model.zero_grad(set_to_none=True)
    logits, balance = model(s["ids"], return_loss=True)
    loss = torch.nn.functional.cross_entropy(logits.flatten(0, 1), s["targets"].flatten()) + balance
    loss.backward()
    # the importance predictor's factor cancels in the renormalisation of the routing weights: its gradient is
    # zero up to rounding, there is nothing to compare
    grads = [p.grad for n, p in model.named_parameters() if p.grad is not None and "importance_predictor" not in n]
    return [loss, *grads, model.pool.fill, model.pool.acc, model.pool.ts]


def _prepare_evict(c, seed):
    g, B, N = _gen(seed), c["batch"], c["context"]
    pool = ops.CachePool([N] * B, c["kv_heads"], c["head_dim"], c["group"], SCHEMES[c["quant"]], _dev())
    _fill_pool(pool, [N] * B, g)
    heavy = torch.rand(B * N, generator=g, device=_dev()) < 0.05
    acc = torch.softmax((torch.randn(B * N, generator=g, device=_dev()) + 4.0 * heavy).view(B, N), dim=-1).view(-1) * 32
    ts = torch.arange(N, dtype=torch.float32, device=_dev()).repeat(B)
    if c["policy"] == "lru":                            # rows were touched in any order
        ts = ts[torch.randperm(B * N, generator=g, device=_dev())].contiguous()
    return dict(case=c, pool=pool, acc=acc, ts=ts, fill=pool.fill.clone(), drop=torch.full_like(pool.fill, N // 2))


def _run_evict(s):
    pool = s["pool"]
    pool.fill.copy_(s["fill"])                          # full again, with the importance the reads have left
    pool.acc.copy_(s["acc"])
    pool.ts.copy_(s["ts"])
    if s["case"]["policy"] == "lru":
        pool.evict(ops.EVICT_LRU, n_evict=s["drop"])
    else:
        pool.evict(ops.EVICT_H2O, heavy_ratio=1 / 16, recent_ratio=1 / 128)
    return [pool.fill, *pool.planes()]


def _prepare_pyramid(c, seed):
    g, dt, L, N = _gen(seed), DTYPES[c["dtype"]], c["layers"], c["tokens"]
    D = c["kv_heads"] * c["head_dim"]
    k, v = (torch.empty(L, N, D, dtype=dt, device=_dev()) for _ in range(2))
    for layer in range(L):
        k[layer], v[layer] = _randn(g, N, D, dtype=dt), _randn(g, N, D, dtype=dt)
    heavy = torch.rand(L, N, generator=g, device=_dev()) < 0.05
    scores = torch.softmax(torch.randn(L, N, generator=g, device=_dev()) + 4.0 * heavy, dim=-1)
    cache = pyramid.PyramidCache(pyramid.linear_keep_budget(N, L), c["kv_heads"], c["head_dim"], group=c["group"],
                                 scheme=SCHEMES[c["quant"]], device=_dev())
    return dict(case=c, k=k, v=v, scores=scores, cache=cache)


def _run_pyramid(s):
    index, kept = s["cache"].compress(s["k"], s["v"], s["scores"])
    return [index, kept, s["cache"].pool.fill, *s["cache"].pool.planes()]


# ---- what a pass cannot do without ------------------------------------------------------------------------------

def _row_bytes(c):
    """Codes, scales and zero points of one cached row of K or of V."""
    D, four = c["kv_heads"] * c["head_dim"], c["quant"].startswith("int4")
    metas = 1 if c["quant"] in ("int8", "int4_sym") else 2
    return D // (2 if four else 1) + D // c["group"] * metas * (2 if four else 4)


def work(case):
    c, kind = case, case["kind"]
    size = 4 if c.get("dtype", "f32") == "f32" else 2
    if kind in ("prefill", "route"):
        D, H, E, k = c["kv_heads"] * c["head_dim"], c["hidden"], c["experts"], c["top_k"]
        T = c["batch"] * c["seq"] if kind == "prefill" else c["tokens"]
        kept = min(T * k, E * _capacity(c), E * c["slots"]) if kind == "prefill" else T * k
        bytes_ = T * H * size + E * H * size + T * E * 4 + T * k * 12 + 2 * T * D * size + kept * (2 * _row_bytes(c) + 8)
        flops = 2.0 * T * H * E
        if kind == "prefill":                           # K read back for the scores, accumulators read and written
            bytes_ += kept * (_row_bytes(c) + 16)
            flops += 2.0 * kept * c["q_heads"] * c["head_dim"]
        return {"bytes": bytes_, "flops": flops}
    if kind == "decode":
        rows = sum(_lengths(c))
        D, q = c["kv_heads"] * c["head_dim"], c["q_heads"] * c["head_dim"]
        return {"bytes": rows * (2 * _row_bytes(c) + 12) + c["batch"] * (2 * D * size + q * (size + 4)),
                "flops": 4.0 * rows * q}
    if kind == "attention":
        B, S, n, H = c["batch"], c["chunk"], c["chunks"], c["hidden"]
        D, q = c["kv_heads"] * c["head_dim"], c["q_heads"] * c["head_dim"]
        cached = B * (c["context"] + (n - 1) * S * n // 2)          # cached rows read, over all chunks
        pairs = B * sum(S * (c["context"] + i * S) + S * (S + 1) / 2 for i in range(n))
        tokens = B * S * n
        weights = H * q * 2 + H * D * 2
        return {"bytes": 4 * weights + 8 * tokens * H + cached * 2 * _row_bytes(c) + tokens * 2 * _row_bytes(c),
                "flops": 2.0 * tokens * weights + 4.0 * pairs * q}
    if kind == "moe":
        T, H, E, V = c["batch"] * c["seq"], c["hidden"], c["experts"], 50257
        dense = E * H * H + 3 * H * H + H * H + V * H               # experts, routers, key projection, vocabulary
        row = 2 * (H + 4)
        rows = sum(c["slots"] - 10 * i for i in range(E))
        scale = 3 if c["train"] else 1                              # forward, and two products of the backward
        return {"bytes": scale * 4 * (dense + T * V) + rows * (H + 4) + 2 * T * row, "flops": scale * 2.0 * T * dense}
    if kind == "evict":
        N, B = c["context"], c["batch"]
        kept = B * (N // 16 + N // 128 if c["policy"] == "h2o" else N - N // 2)
        return {"bytes": B * N * 8 + kept * 2 * (2 * _row_bytes(c) + 8), "flops": 0}
    D = c["kv_heads"] * c["head_dim"]
    kept = sum(pyramid.linear_keep_budget(c["tokens"], c["layers"]))
    return {"bytes": c["layers"] * c["tokens"] * 4 + kept * (2 * D * size + 2 * _row_bytes(c) + 12), "flops": 0}


def tolerance(case):
    """About four times what the paths show against float64, or against the same sums in another order."""
    kind = case["kind"]
    if kind in ("evict", "pyramid"):
        return "exact"                                  # a selection of rows and codes: nothing is rounded twice
    if kind == "route":                                 # probabilities; experts and slots where two of them tie
        return {"rel": 4e-6, "max": 1e-4, "differ": 1e-3}
    if kind == "prefill":                               # importance over 4-bit caches with float32 queries
        return {"rel": 3e-5, "max": 3e-4, "differ": 1e-3}
    if kind == "decode" or case.get("chunk") == 1:      # output over 32768 rows, importance from half precision
        return {"rel": 3e-4, "max": 1.5e-3, "differ": 1e-3}
    if kind == "attention":
        return {"rel": 8e-6, "max": 1e-4, "differ": 1e-3}
    if case["train"]:                                   # gradients, the smallest of them differences of large sums
        return {"rel": 6e-5, "max": 1e-3, "differ": 1e-3}
    return {"rel": 2e-5, "max": 1e-4, "differ": 1e-3}   # moe: float32 products, a code at a rounding edge
