"""NVLLM_ARGMAX_DIRECT: token ids stored by the kernel that picks them, or brought by a copy -- for every kind of model, at every
number of rows the same ids.  It is read once per process, hence the child processes."""
import os
import subprocess
import sys

import pytest

from tests import hybrid_util, latent_util

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import ctypes as C
import sys
import numpy as np
from nvllm_amd import capi
from tests import hybrid_util, test_gpu_thin
lib = capi.load_hip()
lib.init_ops()
f16, f32, latent, hybrid = sys.argv[1:]
for path in (f16, f32):
    for tokens, rows in ((1, 1), (4, 9), (12, 0), (40, 33)):
        ids = np.random.default_rng(tokens).integers(3, 500, 5 + tokens).tolist()
        out = [(7 * k) % tokens for k in range(rows)]
        got, picked = test_gpu_thin.batch(lib, path, 4, ids[:5], ids[5:], out)
        assert picked == (got.argmax(1).tolist() if rows else []), (path, tokens)
for path, in32 in ((latent, 0), (latent, 1), (hybrid, 0), (hybrid, 1)):
    eng = hybrid_util.engine(lib, path, bool(in32), tokens=64)
    for n in (1, 30):
        eng.feed(0, hybrid_util.tokens(n, 130, n), range(n))
        rows, count = eng.feed_run(), C.c_int()
        picked = list(lib.nvllm_last_argmax(C.byref(count))[:n])
        assert count.value == n and picked == rows.argmax(1).tolist(), (path, in32, n)
    eng.feed_end(0)
    eng.close()
"""


@pytest.mark.gpu
@pytest.mark.parametrize("direct", ["0", "1"])
def test_ids_of_every_model(tmp_path, tmp_models, direct):
    paths = [tmp_models("tiny")[0], tmp_models("tiny", dtype="f32", exact16=False)[0], latent_util.model(tmp_path, "heads33")[0], hybrid_util.model(tmp_path, "edges")[0]]
    env = dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_ARGMAX_DIRECT=direct)
    r = subprocess.run([sys.executable, "-c", CHILD, *paths], env=env, capture_output=True, text=True, timeout=150)
    assert r.returncode == 0, r.stderr[-2000:]
