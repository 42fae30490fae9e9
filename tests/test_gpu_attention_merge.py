"""Few sequences with long contexts: the key slices of an item meet in a launch of their own, with one or four waves per row."""
import numpy as np
import pytest

from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,heads,kv_heads,elem,contexts", [
    (16, 4, 2, 4, (700, 33)), (48, 3, 3, 4, (1500,)), (64, 32, 4, 4, (2000, 1, 517)), (80, 2, 1, 4, (1999,)), (128, 2, 2, 4, (900, 16)),
    (64, 32, 4, 2, (2000, 700)), (128, 8, 2, 2, (1300,)), (32, 4, 4, 2, (640, 5)), (64, 8, 8, 4, (40,)),
])
def test_slices_of_long_contexts(hip, hd, heads, kv_heads, elem, contexts):
    rng = np.random.default_rng(hd + len(contexts))
    hip.nvllm_set_kv_elem_bytes(elem)
    try:
        blocks = [-(-c // 16) for c in contexts]
        pool = util.Pool(hip, 16, sum(blocks), 1, kv_heads, hd)
        q = rng.standard_normal((len(contexts), heads * hd)).astype(np.float32)
        rows = [tuple(rng.standard_normal((c, kv_heads * hd)).astype(np.float32) for _ in range(2)) for c in contexts]
        for i, c in enumerate(contexts):
            pool.new_table(blocks[i])
            pool.grow(i, c)
            util.op_kv_write_batch(hip, pool, rows[i][0], rows[i][1], 0, list(range(c)), [i] * c, kv_heads, hd)
        got = util.op_paged_attention_batch(hip, pool, q, 0, [c - 1 for c in contexts], list(range(len(contexts))), max(contexts), heads, kv_heads, hd)
        pool.close()
    finally:
        hip.nvllm_set_kv_elem_bytes(4)
    for i, c in enumerate(contexts):
        k, v = (r.astype(np.float16 if elem == 2 else np.float32).astype(np.float64).reshape(c, kv_heads, hd) for r in rows[i])
        for h in range(heads):
            s = k[:, h * kv_heads // heads] @ q[i, h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
            p = np.exp(s - s.max())
            want = p @ v[:, h * kv_heads // heads] / p.sum()
            # scores carry a few units in the last place (of |s| <= ~6), weights and sums likewise; values are of size one
            np.testing.assert_allclose(got[i, h * hd:(h + 1) * hd], want, atol=4e-6, rtol=0)
