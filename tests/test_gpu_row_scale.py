"""1/rms of a token in the tiles of large batches, to the bit: sums of squares of 32 features each, the even ones and the odd
ones added in order.  Its last bit decides how bf16 activations round, so whatever else a tile does, this order stays."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from nvllm_amd import capi, synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import test_gpu_row_scale
lib = capi.load_hip()
lib.init_ops()
np.save(sys.argv[2], test_gpu_row_scale.logits(lib, sys.argv[1], int(sys.argv[3])))
"""


def write(path, dim, tokens):
    """A layer that adds nothing, one value per 32 features in the embedding, a classifier that picks them out: the logits are
    the values times 1/rms, rounded once.  Returns (the values [token][dim / 32], their features)."""
    rng, groups = np.random.default_rng(dim), dim // 32
    s = synth.ModelShape(dim=dim, hidden_dim=32, n_layers=1, n_heads=dim // 32, n_kv_heads=dim // 32, vocab_size=tokens, max_seq_len=512)
    at = 32 * np.arange(groups) + rng.integers(0, 32, groups)
    values = (rng.choice([-1, 1], (tokens, groups)) * 2.0 ** rng.uniform(-6, 4, (tokens, groups))).astype(np.float16)
    embed, head = np.zeros((tokens, dim), np.float16), np.zeros((tokens, dim), np.float16)
    embed[:, at] = values
    head[np.arange(groups), at] = 1.0
    zeros, ones = (lambda n: np.zeros(n, np.float16)), np.ones(dim, np.float16)
    parts = [embed, ones] + [zeros(dim * dim)] * 4 + [ones] + [zeros(32 * dim)] * 3 + [ones, head]
    with open(path, "wb") as f:
        f.write(s.header())
        for a in parts:
            a.tofile(f)
    return values, at


def logits(lib, path, tokens):
    w, cfg, st = capi.Weights(), capi.Config(), capi.RunState()
    lib.load_model(C.byref(w), C.byref(cfg), path.encode())
    lib.malloc_run_state(C.byref(st), C.byref(cfg))
    mgr = capi.KVCacheManager.in_dll(lib.dll, "g_kv_manager")
    blocks = -(-tokens // 16)
    lib.init_kv_cache_manager(C.byref(mgr), 16, blocks, 1, cfg.n_kv_heads, cfg.head_dim)
    arr = (C.c_int * blocks)(*[lib.alloc_block(C.byref(mgr)) for _ in range(blocks)])
    table = capi.BlockTable(C.cast(arr, capi.c_int_p), blocks)
    tables = (C.POINTER(capi.BlockTable) * 1)(C.pointer(table))
    every = capi.ints(list(range(tokens)))
    lib.transformer_batch(every, tokens, every, capi.ints([0] * tokens), every, tokens, C.byref(cfg), C.byref(st), C.byref(w), tables)
    out = np.ctypeslib.as_array(C.cast(st.logits, capi.c_float_p), shape=(tokens, tokens)).copy()
    lib.free_kv_cache_manager(C.byref(mgr))
    lib.free_run_state(C.byref(st))
    if lib.kind == "hip":
        lib.nvllm_free_model(C.byref(w))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("height", ["0", "4", "6", "9"])   # 0: tiles of 128 features; the others: of 256, that many token blocks
@pytest.mark.parametrize("dim", [2048, 1312, 2176])        # 64, 41 and 68 sums per token: one batch of loads, one value at a time, two batches
def test_order_of_a_tokens_sum_of_squares(tmp_path, dim, height):
    tokens, path, dst = 300, str(tmp_path / "m.bin"), str(tmp_path / "got.npy")
    values, _ = write(path, dim, tokens)
    env = dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_GEMM_WIDE=height)
    r = subprocess.run([sys.executable, "-c", CHILD, path, dst, str(tokens)], env=env, capture_output=True, text=True, timeout=150)
    assert r.returncode == 0, r.stderr[-2000:]
    x = values.astype(np.float32)
    even, odd = np.zeros(tokens, np.float32), np.zeros(tokens, np.float32)
    for j in range(x.shape[1]):   # (a square of an fp16 value is exact in fp32)
        if j % 2:
            odd += x[:, j] * x[:, j]
        else:
            even += x[:, j] * x[:, j]
    rinv = np.float32(1) / np.sqrt((even + odd) / np.float32(dim) + np.float32(1e-5))
    got = np.load(dst)
    np.testing.assert_array_equal(got[:, :x.shape[1]], x * rinv[:, None])
    assert not got[:, x.shape[1]:].any()
