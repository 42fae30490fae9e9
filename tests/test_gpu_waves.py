"""The tiles whose K is dealt to the waves (csrc/gemm_waves.h) at every height, on widths and token counts that end inside a
tile, and K that leaves waves with unequal numbers of steps or none: one projection at a time against the oracle, and whole
passes with every epilogue, in fp16, bf16 rows, bf16 latents with two and with three streams.  The height is read from
the environment once per process, hence a child process per height; the launchers' own rule without it."""
import os
import subprocess
import sys

import numpy as np
import pytest

from nvllm_amd import synth
from tests import dense_tile_child, hybrid_oracle, hybrid_util, latent_oracle, latent_util, test_gpu_wide, util

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOKENS = (256, 300, 433)
HEIGHTS = [1, 2, 3, 4, 5, 6, 7]


def child(code, *args, **env):
    r = subprocess.run([sys.executable, "-c", code, *args], capture_output=True, text=True, timeout=150,
                       env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), **env))
    assert r.returncode == 0, r.stderr[-2000:]


PRODUCTS_CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import dense_tile_child, test_gpu_waves
lib = capi.load_hip()
lib.init_ops()
np.savez(sys.argv[2], **dense_tile_child.run(lib, sys.argv[1], test_gpu_waves.TOKENS))
"""


@pytest.fixture(scope="module")
def wanted(oracle, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("waves") / "m.bin")
    # K of 9, 10 and 25 steps; N of 288, 320, 800 and 1,003
    synth.write_model(path, synth.ModelShape(dim=288, hidden_dim=800, n_layers=1, n_heads=6, n_kv_heads=6, vocab_size=1003, max_seq_len=512), seed=3)
    return path, dense_tile_child.run(oracle, path, TOKENS)


@pytest.mark.gpu
@pytest.mark.parametrize("height", HEIGHTS)
def test_products(wanted, tmp_path, height):
    path, want = wanted
    dst = str(tmp_path / "got.npz")
    child(PRODUCTS_CHILD, path, dst, NVLLM_GEMM_WAVES=str(height))
    got = np.load(dst)
    assert set(got.files) == set(want)
    for key, w in want.items():
        # fp16 weights are exact in both; the activation enters as hi + lo fp16 (~2^-22 relative)
        np.testing.assert_allclose(got[key], w, rtol=0, atol=3e-6 * np.abs(w).max() + 1e-7, err_msg=key)


@pytest.fixture(scope="module")
def passes(oracle, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("waves_passes") / "m.bin")
    synth.write_model(path, synth.ModelShape(dim=256, hidden_dim=800, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=700, max_seq_len=512), seed=5)
    return path, util.run_engine(oracle, path, test_gpu_wide.prompts(), **test_gpu_wide.PASSES)["steps"]


@pytest.mark.gpu
@pytest.mark.parametrize("height,kv_bytes", [(h, 4 if h % 2 else 2) for h in HEIGHTS] + [(None, 2), (None, 4)])
def test_fp16_passes(passes, tmp_path, height, kv_bytes):
    path, want = passes
    dst = str(tmp_path / "got.npz")
    child(test_gpu_wide.CHILD, path, dst, str(kv_bytes), **({"NVLLM_GEMM_WAVES": str(height)} if height else {}))
    got = np.load(dst)
    for i, o in enumerate(want):
        np.testing.assert_array_equal(got[f"sampled{i}"], o["sampled"])
        assert np.abs(got[f"logits{i}"] - o["logits"]).max() < (2e-4 if kv_bytes == 4 else 2e-3)   # the bars of the forward pass


# widths off every tile; query latents of one, two and three steps of K; two streams, and three (the four-stream epilogue)
LATENT = {s: synth.latent_config(288, 203, [(synth.latent_mixer(5, 32, 32, 48, 160, q), ff) for q, ff in ((64, 416), (32, None), (96, 160))], streams=s)
          for s in (2, 3)}
HYBRID = synth.hybrid_config(288, 203, [(hybrid_util.A(6, 2, 48, 64, size=150, keep_first=3, taps=3, rot=16), hybrid_util.E(64, 4, 2, 416)),
                                        (hybrid_util.L(3, 64, 64), 800)])
FOLDER_CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import hybrid_util, latent_util, test_gpu_waves
util = hybrid_util if sys.argv[3] == "hybrid" else latent_util
eng = util.engine(capi.load_hip(), sys.argv[1], False, tokens=704)
got = util.feed_all(eng, [[(0, 300), (1, 257)], [(0, 133)]], test_gpu_waves.sequences())
eng.close()
np.savez(sys.argv[2], **{str(q): rows for q, rows in got.items()})
"""


def sequences():
    return {0: hybrid_util.tokens(433, 203, 1), 1: hybrid_util.tokens(257, 203, 2)}


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    out = {}
    for kind, cfg, util_, oracle_ in [("hybrid", HYBRID, hybrid_util, hybrid_oracle)] + [(f"latent{s}", LATENT[s], latent_util, latent_oracle) for s in LATENT]:
        path, cfg, w = util_.model(tmp_path_factory.mktemp("waves_" + kind), kind, cfg=cfg)
        out[kind] = path, {q: oracle_.forward(cfg, w, seq) for q, seq in sequences().items()}
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("height", HEIGHTS + [None])
@pytest.mark.parametrize("kind", ["hybrid", "latent2", "latent3"])
def test_bf16_passes(folders, tmp_path, kind, height):
    path, want = folders[kind]
    dst = str(tmp_path / "got.npz")
    child(FOLDER_CHILD, path, dst, kind, **({"NVLLM_GEMM_WAVES": str(height)} if height else {}))
    got = np.load(dst)
    for q, o in want.items():
        assert hybrid_util.error(got[str(q)], o) < hybrid_util.limit(False), q   # the bar of the designs' whole passes


# Passes of 65 to 255 tokens: gated pairs so wide that groups of 64 tokens are more workgroups than CUs, and narrow
# projections past 128 tokens (csrc/gemm_common.h, gemm_leaves_streaming)
@pytest.mark.gpu
@pytest.mark.parametrize("kv_bytes", [4, 2])
def test_between_decode_and_prompts_fp16(hip, oracle, tmp_path, kv_bytes):
    path = str(tmp_path / "m.bin")
    synth.write_model(path, synth.ModelShape(dim=256, hidden_dim=5632, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=700, max_seq_len=512), seed=7)
    for chunk in (65, 129, 193, 255):
        kw = dict(n_new=2, collect_logits=True, chunk_size=chunk, temperature=0.0)
        want = util.run_engine(oracle, path, synth.make_requests(1, 255, 256, 700, seed=chunk), **kw)["steps"]
        hip.nvllm_set_kv_elem_bytes(kv_bytes)
        try:
            got = util.run_engine(hip, path, synth.make_requests(1, 255, 256, 700, seed=chunk), **kw)["steps"]
        finally:
            hip.nvllm_set_kv_elem_bytes(4)
        for g, o in zip(got, want):
            np.testing.assert_array_equal(g["sampled"], o["sampled"])
            assert np.abs(g["logits"] - o["logits"]).max() < (2e-4 if kv_bytes == 4 else 2e-3)   # the bars of the forward pass


@pytest.mark.gpu
def test_between_decode_and_prompts_bf16(hip, tmp_path):
    cfg = synth.latent_config(256, 203, [(synth.latent_mixer(4, 32, 32, 32, 64, 96), 5632)] * 2, streams=2)
    path, cfg, w = latent_util.model(tmp_path, "between", cfg=cfg)
    seq = hybrid_util.tokens(700, 203, 3)
    want = latent_oracle.forward(cfg, w, seq)
    eng = latent_util.engine(hip, path, False, tokens=704)
    got = latent_util.feed_all(eng, [[(0, n)] for n in (65, 255, 129, 193, 58)], {0: seq})[0]
    eng.close()
    assert latent_util.error(got, want) < latent_util.limit(False)
