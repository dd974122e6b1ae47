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
