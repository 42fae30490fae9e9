"""A pass that fills the staging of its integer arrays to the last number, here with a sequence of a very high id: prompt portions of
the Suselorn design, whose formed keys and values (csrc/latent_prompt.hip) have a list of pages there, do without."""
import os
import subprocess
import sys

import numpy as np
import pytest

from nvllm_amd import synth
from tests import latent_oracle as O
from tests import latent_util as U
from tests.test_gpu_latent_prompt import ROOT

pytestmark = pytest.mark.gpu
STAGING, T = 1 << 20, 256
CHILD = """
import ctypes as C
import sys
import numpy as np
from nvllm_amd import capi
from tests import latent_util as U, test_gpu_latent_staging as me
hip, T = capi.load_hip(), me.T
hip.nvllm_set_compute_dtype(capi.COMPUTE_BF16)
hip.nvllm_set_logits_mode(0)
w, cfg, st = capi.Weights(), capi.Config(), capi.RunState()
hip.load_model(C.byref(w), C.byref(cfg), sys.argv[1].encode())
cfg.max_seq_len = T
hip.malloc_run_state(C.byref(st), C.byref(cfg))
mgr = capi.KVCacheManager.in_dll(hip.dll, "g_kv_manager")
hip.nvllm_set_kv_elem_bytes(2)
hip.nvllm_init_model_kv(C.byref(mgr), 16, T // 16, C.byref(cfg), C.byref(w))
# tokens, positions, ids and cache rows; output row; a table of T / 16 blocks; T / 32 items of attention of four numbers; 64 to spare
top = me.STAGING - (4 * T + 1 + T // 16 + T // 32 * 4 + 64)
at = (C.c_int * (T // 16))(*[hip.alloc_block(C.byref(mgr)) for _ in range(T // 16)])
table = capi.BlockTable(C.cast(at, capi.c_int_p), T // 16)
rows = []
for n_ids in (8, top):
    tables = (C.POINTER(capi.BlockTable) * n_ids)()
    tables[n_ids - 1] = C.pointer(table)
    hip.transformer_batch(capi.ints(U.tokens(T, cfg.vocab_size, 1)), T, capi.ints(range(T)), capi.ints([n_ids - 1] * T), capi.ints([T - 1]), 1,
                          C.byref(cfg), C.byref(st), C.byref(w), tables)
    rows.append(np.ctypeslib.as_array(C.cast(st.logits, capi.c_float_p), shape=(cfg.vocab_size,)).copy())
np.save(sys.argv[2], rows)
"""


def test_no_room_for_the_pages_of_prompts(tmp_path):
    cfg = synth.latent_config(64, 130, [(synth.latent_mixer(4, 64, 32, 64, 64, 32), 40)] * 2, streams=2)
    path, cfg, w = U.model(tmp_path, "staging", seed=5, cfg=cfg)
    dst = str(tmp_path / "rows.npy")
    r = subprocess.run([sys.executable, "-c", CHILD, path, dst], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_LATENT_EXPAND="1"))
    assert r.returncode == 0, r.stderr[-2000:]
    want = O.forward(cfg, w, U.tokens(T, 130, 1))[-1:]
    for row in np.load(dst):
        assert U.error(row[None], want) < U.limit(False)
