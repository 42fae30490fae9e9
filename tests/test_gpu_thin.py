"""Passes on either side of the line between the few-token projections and the tiles of 16 and more: a batch of n one-token
rows at widths whose K ends inside a wave's ring, a vocabulary that ends inside a row block, both pool formats; and passes
whose layers and whose classifier lie on different sides of it."""
import ctypes as C

import numpy as np
import pytest

from nvllm_amd import capi, synth
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 5, 6, 7])
@pytest.mark.parametrize("kv_bytes", [4, 2])
@pytest.mark.parametrize("shape", [
    dict(dim=96, hidden_dim=224, n_layers=2, n_heads=2, n_kv_heads=2, vocab_size=1003),        # 3 and 7 tiles of K
    dict(dim=512, hidden_dim=2080, n_layers=1, n_heads=8, n_kv_heads=2, vocab_size=16500),     # more row blocks than 4 per CU in the classifier
])
def test_few_rows(hip, oracle, tmp_path, n, kv_bytes, shape):
    s = synth.ModelShape(max_seq_len=64, **shape)
    path = str(tmp_path / "m.bin")
    synth.write_model(path, s, seed=n)
    prompts = synth.make_requests(n, 3, 20, s.vocab_size, seed=n + 1)
    kw = dict(n_new=6, collect_logits=True, chunk_size=5, temperature=0.0)
    want = util.run_engine(oracle, path, prompts, **kw)
    before = hip.nvllm_get_kv_elem_bytes()
    hip.nvllm_set_kv_elem_bytes(kv_bytes)
    try:
        got = util.run_engine(hip, path, prompts, **kw)
    finally:
        hip.nvllm_set_kv_elem_bytes(before)
    np.testing.assert_array_equal(got["trace"], want["trace"])
    assert n in {len(st["tokens"]) for st in got["steps"]}   # a pass of just that many tokens
    for g, o in zip(got["steps"], want["steps"]):
        np.testing.assert_array_equal(g["sampled"], o["sampled"])
        # the bars of the forward pass: exact pool rows, fp16 pool rows
        assert np.abs(g["logits"] - o["logits"]).max() < (2e-4 if kv_bytes == 4 else 2e-3)


@pytest.mark.parametrize("n", [1, 2, 3])
@pytest.mark.parametrize("shape", [
    dict(dim=2112, hidden_dim=4128, n_layers=1, n_heads=33, n_kv_heads=3, vocab_size=16500),   # 66 and 129 tiles of K: every wave's ring and one or two tiles more
    dict(dim=2048, hidden_dim=4096, n_layers=1, n_heads=32, n_kv_heads=4, vocab_size=16400),   # the fewest tiles
])
def test_activations_laid_out_once(hip, oracle, tmp_path, n, shape):
    """One and two rows at widths whose projections lay their activations out in LDS, and three rows, which do not."""
    test_few_rows(hip, oracle, tmp_path, n, 4, shape)


@pytest.mark.parametrize("n", [1, 2, 3])
@pytest.mark.parametrize("kv_bytes", [4, 2])
@pytest.mark.parametrize("shape", [
    dict(dim=2048, hidden_dim=4096, n_layers=1, n_heads=32, n_kv_heads=32, vocab_size=16400),  # q/k/v and gate/up: the fewest tiles
    dict(dim=1024, hidden_dim=3104, n_layers=1, n_heads=16, n_kv_heads=4, vocab_size=500),     # w_down on 16 waves: a tile more than the fewest
    dict(dim=512, hidden_dim=8192, n_layers=1, n_heads=8, n_kv_heads=4, vocab_size=500),       # two tokens: a lap to the last value; 8,224 are one value of every thread too many
    dict(dim=512, hidden_dim=8224, n_layers=1, n_heads=8, n_kv_heads=4, vocab_size=500),
    dict(dim=1024, hidden_dim=512, n_layers=1, n_heads=16, n_kv_heads=4, vocab_size=16),       # the classifier on 16 waves, with the norm: one block, two tiles of K a wave
    dict(dim=5120, hidden_dim=480, n_layers=1, n_heads=40, n_kv_heads=8, vocab_size=500),      # q/k/v and wo on 8 waves: two laps, the second one ragged
])
def test_lines_of_the_rule_for_activations_laid_out_once(hip, oracle, tmp_path, n, kv_bytes, shape):
    test_few_rows(hip, oracle, tmp_path, n, kv_bytes, shape)


@pytest.mark.parametrize("n", [1, 2])
@pytest.mark.parametrize("kv_bytes", [4, 2])
def test_activations_of_a_7b_layer(hip, oracle, tmp_path, n, kv_bytes):
    """768 workgroups of q/k/v, 688 of gate/up, w_down of 344 tiles on 16 waves (one row)."""
    test_few_rows(hip, oracle, tmp_path, n, kv_bytes, dict(dim=4096, hidden_dim=11008, n_layers=1, n_heads=32, n_kv_heads=32, vocab_size=500))


def batch(lib, path, kv_bytes, history, tokens, out):
    """Logits rows (and the library's token ids) of one pass of one sequence behind `history`."""
    w, cfg, st = capi.Weights(), capi.Config(), capi.RunState()
    lib.load_model(C.byref(w), C.byref(cfg), path.encode())
    lib.malloc_run_state(C.byref(st), C.byref(cfg))
    if lib.kind == "hip":
        before = lib.nvllm_get_kv_elem_bytes()
        lib.nvllm_set_kv_elem_bytes(kv_bytes)
    mgr = capi.KVCacheManager.in_dll(lib.dll, "g_kv_manager")
    lib.init_kv_cache_manager(C.byref(mgr), 16, 4, cfg.n_layers, cfg.n_kv_heads, cfg.head_dim)
    arr = (C.c_int * 4)(*[lib.alloc_block(C.byref(mgr)) for _ in range(4)])
    table = capi.BlockTable(C.cast(arr, capi.c_int_p), 4)
    tables = (C.POINTER(capi.BlockTable) * 1)(C.pointer(table))
    for part, at, rows in ((history, 0, [0]), (tokens, len(history), out)):
        n = len(part)
        lib.transformer_batch(capi.ints(part), n, capi.ints(range(at, at + n)), capi.ints([0] * n), capi.ints(rows), len(rows), C.byref(cfg), C.byref(st),
                              C.byref(w), tables)
    V = cfg.vocab_size
    logits = np.ctypeslib.as_array(C.cast(st.logits, capi.c_float_p), shape=(len(out), V)).copy()
    ids = None
    if lib.kind == "hip":
        n = C.c_int()
        ids = list(lib.nvllm_last_argmax(C.byref(n))[:len(out)])
        assert n.value == len(out)
        lib.nvllm_set_kv_elem_bytes(before)
    lib.free_kv_cache_manager(C.byref(mgr))
    lib.free_run_state(C.byref(st))
    if lib.kind == "hip":
        lib.nvllm_free_model(C.byref(w))
    return logits, ids


@pytest.mark.parametrize("kv_bytes", [4, 2])
@pytest.mark.parametrize("tokens,rows", [(1, 7), (1, 17), (3, 8), (6, 7), (6, 17), (6, 6), (3, 0), (9, 5), (17, 1), (20, 6)])
def test_output_rows_that_repeat(hip, oracle, tmp_models, tokens, rows, kv_bytes):
    """Few tokens and more output rows than that (eight samples of a prompt's last token), many tokens and a few rows of them
    out of order, and nobody's row."""
    path, shape = tmp_models("tiny")
    rng = np.random.default_rng(100 * tokens + rows)
    out = [int(i) for i in rng.integers(0, tokens, rows)]
    ids = rng.integers(3, shape.vocab_size, 11 + tokens).tolist()
    want, _ = batch(oracle, path, 4, ids[:11], ids[11:], out)
    got, picked = batch(hip, path, kv_bytes, ids[:11], ids[11:], out)
    assert picked == want.argmax(1).tolist() if rows else picked == []
    if rows:
        assert np.abs(got - want).max() < (2e-4 if kv_bytes == 4 else 2e-3)   # the bars of the forward pass
