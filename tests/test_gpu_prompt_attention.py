"""Attention of prompt portions over fp16 pages: batches that take the kernel of 64 columns a workgroup, against plain float64.

Portions begin and end inside runs, blocks of 64 keys and halves of them; single tokens and short ends ride in the same launch.
"""
import numpy as np
import pytest

from tests import util

pytestmark = pytest.mark.gpu


def want(q, k, v, first):
    """q [n, hd] at positions first .., k and v [m, hd]; weights and sums in float64."""
    s = q.astype(np.float64) @ k.T / np.sqrt(q.shape[1])
    s[np.arange(len(k))[None] > first + np.arange(len(q))[:, None]] = -np.inf
    p = np.exp(s - s.max(1, keepdims=True))
    return p @ v / p.sum(1, keepdims=True)


@pytest.mark.parametrize("scale", [1.0, 30.0])   # (scores far apart: the running maximum rises late, weights fall below fp16's range)
@pytest.mark.parametrize("hd,heads,kv_heads", [(64, 16, 4), (64, 32, 4), (64, 8, 8), (128, 16, 16), (128, 16, 2), (32, 16, 1), (96, 12, 4)])
def test_portions(hip, hd, heads, kv_heads, scale):
    # (first position, tokens): a run's remainder of 1, ends on and around 32 and 64 keys, rows of single tokens, a portion too short
    parts = [(0, 577), (63, 129), (0, 1), (700, 1), (31, 65), (5, 2), (128, 64), (15, 500), (64, 1)]
    r = np.random.default_rng(hd + heads)
    hip.nvllm_set_kv_elem_bytes(2)
    try:
        pool = util.Pool(hip, 16, sum(-(-(a + n) // 16) for a, n in parts), 1, kv_heads, hd)
        rows = [tuple(r.standard_normal((a + n, kv_heads * hd)).astype(np.float32) for _ in range(2)) for a, n in parts]
        q = (scale * r.standard_normal((sum(n for _, n in parts), heads * hd))).astype(np.float32)
        pos, seq = [], []
        for i, (a, n) in enumerate(parts):
            pool.new_table(-(-(a + n) // 16))
            pool.grow(i, a + n)
            util.op_kv_write_batch(hip, pool, rows[i][0], rows[i][1], 0, list(range(a + n)), [i] * (a + n), kv_heads, hd)
            pos += list(range(a, a + n))
            seq += [i] * n
        got = util.op_paged_attention_batch(hip, pool, q, 0, pos, seq, max(pos) + 1, heads, kv_heads, hd)
        pool.close()
    finally:
        hip.nvllm_set_kv_elem_bytes(4)
    at = 0
    for i, (a, n) in enumerate(parts):
        k, v = (x.astype(np.float16).astype(np.float64).reshape(-1, kv_heads, hd) for x in rows[i])
        for h in range(heads):
            w = want(q[at:at + n, h * hd:(h + 1) * hd], k[:, h * kv_heads // heads], v[:, h * kv_heads // heads], a)
            # scores, weights and sums carry a few units in the last place, scores of some hundreds that many times more
            np.testing.assert_allclose(got[at:at + n, h * hd:(h + 1) * hd], w, atol=4e-6 * max(1.0, scale), rtol=0, err_msg="portion %d head %d" % (i, h))
        at += n
