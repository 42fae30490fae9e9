"""Passes on either side of the line between the few-token projections and the tiles of 16 and more: a batch of n one-token
rows at widths whose K ends inside a wave's ring, a vocabulary that ends inside a row block, both pool formats."""
import numpy as np
import pytest

from nvllm_amd import synth
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
    assert min(len(st["tokens"]) for st in got["steps"]) <= 8
    for g, o in zip(got["steps"], want["steps"]):
        np.testing.assert_array_equal(g["sampled"], o["sampled"])
        # the bars of the forward pass: exact pool rows, fp16 pool rows
        assert np.abs(g["logits"] - o["logits"]).max() < (2e-4 if kv_bytes == 4 else 2e-3)
