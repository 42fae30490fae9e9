"""Attention around the lengths from which key slices meet in a launch of their own, and from which a window is cut into slices."""
import numpy as np
import pytest

from tests import util
from tests.test_gpu_hybrid_ops import filled, reference
from tests.test_gpu_latent_ops import rng, rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("longest", [16, 304, 305, 320, 321, 400, 480, 650, 1040])
@pytest.mark.parametrize("hd,heads,kv_heads,elem", [(64, 16, 4, 4), (48, 4, 4, 4), (64, 16, 4, 2), (128, 4, 2, 2)])
def test_rows(hip, hd, heads, kv_heads, elem, longest):
    contexts = [longest, 1, 17, max(1, longest - 100)] * (5 if elem == 4 else 2)   # 16 to 80 items
    hip.nvllm_set_kv_elem_bytes(elem)
    try:
        check_rows(hip, hd, heads, kv_heads, elem, longest, contexts)
    finally:
        hip.nvllm_set_kv_elem_bytes(4)


def check_rows(hip, hd, heads, kv_heads, elem, longest, contexts):
    r = np.random.default_rng(longest + hd)
    pool = util.Pool(hip, 16, sum(-(-c // 16) for c in contexts), 1, kv_heads, hd)
    q = r.standard_normal((len(contexts), heads * hd)).astype(np.float32)
    rows = [tuple(r.standard_normal((c, kv_heads * hd)).astype(np.float32) for _ in range(2)) for c in contexts]
    for i, c in enumerate(contexts):
        pool.new_table(-(-c // 16))
        pool.grow(i, c)
        util.op_kv_write_batch(hip, pool, rows[i][0], rows[i][1], 0, list(range(c)), [i] * c, kv_heads, hd)
    got = util.op_paged_attention_batch(hip, pool, q, 0, [c - 1 for c in contexts], list(range(len(contexts))), longest, heads, kv_heads, hd)
    pool.close()
    for i, c in enumerate(contexts):
        k, v = (x.astype(np.float16 if elem == 2 else np.float32).astype(np.float64).reshape(c, kv_heads, hd) for x in rows[i])
        for h in range(heads):
            s = k[:, h * kv_heads // heads] @ q[i, h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
            p = np.exp(s - s.max())
            # the bar of test_gpu_attention_merge.py: scores, weights and sums carry a few units in the last place
            np.testing.assert_allclose(got[i, h * hd:(h + 1) * hd], p @ v[:, h * kv_heads // heads] / p.sum(), atol=4e-6, rtol=0)


@pytest.mark.parametrize("length", [1, 33, 1503, 1504, 1505, 1600, 2500])   # (six pairs of pages for eight waves: 1,536 keys, 32 of them for the window's ends)
@pytest.mark.parametrize("dim,size", [(64, 512), (64, 1 << 30), (128, 1 << 30)])
def test_windowed_tokens(hip, dim, size, length):
    pool, kv = filled(hip, 2, dim, 64, 2, 16, [length, 5], dim)
    q = rounded(rng(length).standard_normal((2, 8, dim)), 2)
    got = pool.attend([0, 1], [length - 1, 4], q, dim ** -0.5, 20.0, size, 4)
    want = reference(kv, q, [length - 1, 4], [0, 1], dim ** -0.5, 20.0, size, 4)
    assert np.abs(got - want).max() < 1.2e-2 * np.abs(want).max()   # the bar of test_gpu_hybrid_ops.py
    pool.close()
