"""Attention of prompt portions over fp16 pages: batches that take the kernel of 64 columns a workgroup, against plain float64.

Portions begin and end inside runs, blocks of 64 keys and halves of them; single tokens and short ends ride in the same launch.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

from nvllm_amd import synth
from tests import test_gpu_wide, util

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
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


@pytest.mark.parametrize("hd,heads,kv_heads", [(32, 8, 8), (32, 8, 1), (64, 6, 3), (96, 4, 4), (96, 4, 1), (128, 4, 4), (128, 4, 2)])
def test_passes_store_activation_tiles(oracle, tmp_path, hd, heads, kv_heads):
    """Whole passes, whose next projection reads the results as tiles of two planes: against the oracle, and against the attention of 16 columns (the
    environment, read once per process, lets one item be enough, or none)."""
    path = str(tmp_path / "m.bin")
    synth.write_model(path, synth.ModelShape(dim=hd * heads, hidden_dim=416, n_layers=2, n_heads=heads, n_kv_heads=kv_heads, vocab_size=700, max_seq_len=512), seed=hd)
    want = util.run_engine(oracle, path, test_gpu_wide.prompts(), **test_gpu_wide.PASSES)["steps"]
    got = []
    for items in ("1", "0"):
        dst = str(tmp_path / ("got%s.npz" % items))
        r = subprocess.run([sys.executable, "-c", test_gpu_wide.CHILD, path, dst, "2"], capture_output=True, text=True, timeout=110,
                           env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_ATTN_LONG=items))
        assert r.returncode == 0, r.stderr[-2000:]
        got.append(np.load(dst))
    apart = 0.0
    for i, o in enumerate(want):
        np.testing.assert_array_equal(got[0][f"sampled{i}"], o["sampled"])
        assert np.abs(got[0][f"logits{i}"] - o["logits"]).max() < 2e-3   # the bar of the forward pass over an fp16 pool
        apart = max(apart, float(np.abs(got[0][f"logits{i}"] - got[1][f"logits{i}"]).max()))
    assert 0 < apart < 2e-4   # (other sums, so some bit differs; the bar of the pass over an fp32 pool)


ERROR_CHILD = """
import sys
from nvllm_amd import capi
from tests import test_gpu_prompt_attention as T
lib = capi.load_hip()
lib.init_ops()
print("error", T.error(lib, *map(int, sys.argv[1:])))
"""


def error(hip, hd, heads, kv_heads):
    """2-norm of the results' distance from float64 over that of the results; queries of size 1, where the sums' roundings are most of it."""
    parts, off, size = [(512, 300), (0, 300)], 0.0, 0.0
    hip.nvllm_set_kv_elem_bytes(2)
    for seed in range(3):
        r = np.random.default_rng(seed)
        pool = util.Pool(hip, 16, sum(-(-(a + n) // 16) for a, n in parts), 1, kv_heads, hd)
        rows = [tuple(r.standard_normal((a + n, kv_heads * hd)).astype(np.float32) for _ in range(2)) for a, n in parts]
        q = r.standard_normal((sum(n for _, n in parts), heads * hd)).astype(np.float32)
        pos, seq = [], []
        for i, (a, n) in enumerate(parts):
            pool.new_table(-(-(a + n) // 16))
            pool.grow(i, a + n)
            util.op_kv_write_batch(hip, pool, rows[i][0], rows[i][1], 0, list(range(a + n)), [i] * (a + n), kv_heads, hd)
            pos += list(range(a, a + n))
            seq += [i] * n
        got = util.op_paged_attention_batch(hip, pool, q, 0, pos, seq, max(pos) + 1, heads, kv_heads, hd)
        pool.close()
        at = 0
        for i, (a, n) in enumerate(parts):
            k, v = (x.astype(np.float16).astype(np.float64).reshape(-1, kv_heads, hd) for x in rows[i])
            for h in range(heads):
                w = want(q[at:at + n, h * hd:(h + 1) * hd], k[:, h * kv_heads // heads], v[:, h * kv_heads // heads], a)
                off, size = off + ((got[at:at + n, h * hd:(h + 1) * hd] - w) ** 2).sum(), size + (w ** 2).sum()
            at += n
    return float(np.sqrt(off / size))


@pytest.mark.parametrize("hd,heads,kv_heads", [(32, 8, 2), (64, 8, 2), (96, 8, 2), (128, 8, 2), (128, 8, 8)])
def test_no_further_from_64_bits_than_sixteen_columns(hd, heads, kv_heads):
    got = []
    for items in ("1", "0"):
        r = subprocess.run([sys.executable, "-c", ERROR_CHILD, str(hd), str(heads), str(kv_heads)], capture_output=True, text=True, timeout=110,
                           env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_ATTN_LONG=items))
        assert r.returncode == 0, r.stderr[-2000:]
        got.append(float(r.stdout.split()[-1]))
    assert got[0] < got[1], got
