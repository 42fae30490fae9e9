"""Streaming projections where a wave's K-steps are fewer than, as many as and a few more than it has in flight, and where a token has
more sums of squares than are held over the K loop; and the token ids that the classifier's blocks of fp32 models leave."""
import numpy as np
import pytest

from nvllm_amd import synth
from tests import test_gpu_thin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [9, 20, 40, 59])   # one, two and four token blocks a tile, the last of them ragged
@pytest.mark.parametrize("shape", [
    dict(dim=192, hidden_dim=480, n_heads=3, n_kv_heads=3),       # 6 and 15 tiles of K for eight waves
    dict(dim=1056, hidden_dim=992, n_heads=33, n_kv_heads=3),     # four steps a wave and five, three and four
    dict(dim=2048, hidden_dim=2304, n_heads=32, n_kv_heads=4),    # eight steps a wave, nine
    dict(dim=2112, hidden_dim=2368, n_heads=33, n_kv_heads=3),    # eight or nine; 66 sums of squares
])
def test_steps_around_the_rings(hip, oracle, tmp_path, T, shape):
    s = synth.ModelShape(max_seq_len=64, n_layers=1, vocab_size=500, **shape)
    path = str(tmp_path / "m.bin")
    synth.write_model(path, s, seed=T)
    ids = np.random.default_rng(T).integers(3, 500, 5 + T).tolist()
    want, _ = test_gpu_thin.batch(oracle, path, 4, ids[:5], ids[5:], list(range(T)))
    got, picked = test_gpu_thin.batch(hip, path, 4, ids[:5], ids[5:], list(range(T)))
    assert np.abs(got - want).max() < 2e-4   # the bar of the forward pass over exact pool rows
    assert picked == got.argmax(1).tolist()


@pytest.mark.parametrize("T,rows", [(1, 1), (9, 9), (40, 3), (59, 59)])
@pytest.mark.parametrize("dim,vocab", [(96, 1003), (288, 16401)])   # one block more than full tiles have
def test_ids_of_fp32_models(hip, tmp_path, T, rows, dim, vocab):
    s = synth.ModelShape(dim=dim, hidden_dim=2 * dim, n_layers=1, n_heads=6, n_kv_heads=6, vocab_size=vocab, max_seq_len=64)
    path = str(tmp_path / "m.bin")
    synth.write_model(path, s, seed=T, dtype="f32", shared=True, exact16=False)
    ids = np.random.default_rng(T).integers(3, vocab, 5 + T).tolist()
    out = [(7 * k) % T for k in range(rows)]
    got, picked = test_gpu_thin.batch(hip, path, 4, ids[:5], ids[5:], out)
    assert picked == got.argmax(1).tolist()
