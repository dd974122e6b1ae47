"""GPU parity of the launch shapes small calls take: few caches, short caches, few blocks."""
import numpy as np
import pytest

import pikv_oracle as O
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
