"""Streaming projections where a wave's K-steps are fewer than, as many as and a few more than it has in flight, and where a token has
more sums of squares than are held over the K loop; and the token ids that the classifier's blocks of fp32 models leave."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from nvllm_amd import capi, synth
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


def fp32_model(path, T, dim, vocab, max_seq_len=64):
    """An fp32 model of one layer; returns its token rows, the classifier's as well, as an array over the file."""
    s = synth.ModelShape(dim=dim, hidden_dim=2 * dim, n_layers=1, n_heads=max(1, dim // 48), n_kv_heads=max(1, dim // 48), vocab_size=vocab, max_seq_len=max_seq_len)
    synth.write_model(path, s, seed=T, dtype="f32", shared=True, exact16=False)
    return np.memmap(path, np.float32, "r+", len(s.header()), (vocab, dim))


def scan(row):
    """The reference's pick (sampler.c:86-97)."""
    best = 0
    for i in np.flatnonzero(row >= (row[0] if row[0] == row[0] else np.inf)):
        if row[i] > row[best]:
            best = int(i)
    return best


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


@pytest.mark.parametrize("T,rows", [(1, 1), (9, 9), (40, 3), (59, 59)])
@pytest.mark.parametrize("dim,vocab", [(96, 1003), (288, 16385)])   # 63 blocks; 1,025, whose last tile of two is half empty (16,401 words have 1,026)
def test_ids_where_the_last_tile_is_half_empty(hip, tmp_path, T, rows, dim, vocab):
    path = str(tmp_path / "m.bin")
    fp32_model(path, T, dim, vocab)
    ids = np.random.default_rng(T).integers(3, vocab, 5 + T).tolist()
    got, picked = test_gpu_thin.batch(hip, path, 4, ids[:5], ids[5:], [(7 * k) % T for k in range(rows)])
    assert picked == got.argmax(1).tolist()


@pytest.mark.parametrize("nan_row", [0, 3])
@pytest.mark.parametrize("T,rows", [(1, 1), (9, 9), (40, 33)])
@pytest.mark.parametrize("dim,vocab", [(96, 1003), (288, 16385)])
def test_ids_of_fp32_models_with_ties_nan_and_infinities(hip, tmp_path, T, rows, dim, vocab, nan_row):
    """Classifier rows repeat every 37 indices, so that each maximum is attained in every tile; one row is NaN, which never wins but
    at index 0, where nothing displaces it; one is infinite, with a sign that depends on the token."""
    path = str(tmp_path / "m.bin")
    head = fp32_model(path, T, dim, vocab)
    head[:] = head[np.arange(vocab) % 37]
    head[nan_row] = np.nan
    head[vocab - 2] = 0
    head[vocab - 2, 0] = np.inf
    head.flush()
    ids = np.random.default_rng(T).integers(4, vocab - 2, 5 + T).tolist()
    got, picked = test_gpu_thin.batch(hip, path, 4, ids[:5], ids[5:], [(7 * k) % T for k in range(rows)])
    assert np.isnan(got[:, nan_row]).all() and np.isinf(got[:, vocab - 2]).all()
    assert picked == [scan(r) for r in got]


def test_ids_beyond_what_fp32_holds(hip, tmp_path):
    """From 16,777,217 words on an index in fp32 is not every index: the rows are scanned for it."""
    path, small, dim, vocab = str(tmp_path / "m.bin"), str(tmp_path / "small.bin"), 32, (1 << 24) + 32
    few = np.array(fp32_model(small, 1, dim, 1 << 14, max_seq_len=16))
    shape = synth.ModelShape(dim=dim, hidden_dim=2 * dim, n_layers=1, n_heads=1, n_kv_heads=1, vocab_size=vocab, max_seq_len=16)
    with open(small, "rb") as f, open(path, "wb") as out:
        f.seek(len(shape.header()) + few.nbytes)
        out.write(shape.header())
        for _ in range(1 << 10):
            out.write((few / np.float32(64)).data)
        out.write(few[:32].data)   # the maximum is one of the last 32
        out.write(f.read())
    got, picked = test_gpu_thin.batch(hip, path, 4, [5, 6], list(range(7, 19)), list(range(12)))
    want = got.argmax(1)
    assert (want >= 1 << 24).all() and (want % 2 == 1).any()
    assert picked == want.tolist()


def pair_room_of_one_row(folder):
    """Bytes that the first pass of one row takes on the GPU and keeps (run in a process of its own: what a pass keeps only grows)."""
    hip, vocab = capi.load_hip(), 1 << 20
    hip.init_ops()
    free, total = C.c_size_t(), C.c_size_t()
    seen = []
    for words in (500, vocab):
        path = os.path.join(folder, "m%d.bin" % words)
        fp32_model(path, 1, 32, words)
        test_gpu_thin.batch(hip, path, 4, [5], [6], [0])
        assert C.CDLL("libamdhip64.so").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        seen.append(free.value)
    return seen[0] - seen[1]


def test_pairs_have_room_for_64_rows_from_the_first_row_on(hip, tmp_path):
    """A batch that grows row by row does not allocate them again and again."""
    code = "from tests import test_gpu_stream_rings as t; print('ROOM', t.pair_room_of_one_row(%r))" % str(tmp_path)
    out = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    assert int(out.stdout.split("ROOM")[1]) >= 64 * (1 << 16) * 8
