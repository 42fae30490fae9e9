"""The 256-feature tiles (csrc/gemm_wide.h) at every height, on widths and token counts that end inside a tile, and K that
ends inside a turn of the ring: one projection at a time against the oracle, and whole passes with every epilogue.  The
height is read from the environment once per process, hence a child process per height.  In bf16 too, and by the launchers'
own rules."""
import os
import subprocess
import sys

import numpy as np
import pytest

from nvllm_amd import synth
from tests import dense_tile_child, hybrid_oracle, hybrid_util, latent_oracle, latent_util, test_gpu_row_scale, util

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOKENS = (256, 300, 433)


@pytest.fixture(scope="module")
def wanted(oracle, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("wide") / "m.bin")
    # K of 9, 10 and 25 steps; N of 288, 320, 800 and 1,003
    synth.write_model(path, synth.ModelShape(dim=288, hidden_dim=800, n_layers=1, n_heads=6, n_kv_heads=6, vocab_size=1003, max_seq_len=512), seed=3)
    return path, dense_tile_child.run(oracle, path, TOKENS)


@pytest.mark.gpu
@pytest.mark.parametrize("height", [4, 6, 9])
def test_every_height_of_the_wide_tiles(wanted, tmp_path, height):
    path, want = wanted
    dst = str(tmp_path / "got.npz")
    env = dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""))
    env["NVLLM_GEMM_WIDE"] = str(height)
    r = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "dense_tile_child.py"), path, dst, ",".join(map(str, TOKENS))], env=env,
                       capture_output=True, text=True, timeout=150)
    assert r.returncode == 0, r.stderr[-2000:]
    got = np.load(dst)
    assert set(got.files) == set(want)
    for key, w in want.items():
        # fp16 weights are exact in both; the activation enters as hi + lo fp16 (~2^-22 relative)
        np.testing.assert_allclose(got[key], w, rtol=0, atol=3e-6 * np.abs(w).max() + 1e-7, err_msg=key)


PASSES = dict(n_new=3, collect_logits=True, chunk_size=280, temperature=0.0)
CHILD = """
import sys
import numpy as np
from nvllm_amd import capi, synth
from tests import test_gpu_wide, util
lib = capi.load_hip()
lib.nvllm_set_kv_elem_bytes(int(sys.argv[3]))
steps = util.run_engine(lib, sys.argv[1], test_gpu_wide.prompts(), **test_gpu_wide.PASSES)["steps"]
np.savez(sys.argv[2], **{k + str(i): s[k] for i, s in enumerate(steps) for k in ("sampled", "logits")})
"""


def prompts():
    return synth.make_requests(2, 300, 301, 700, seed=6)


@pytest.fixture(scope="module")
def passes(oracle, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("wide_passes") / "m.bin")
    synth.write_model(path, synth.ModelShape(dim=256, hidden_dim=800, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=700, max_seq_len=512), seed=5)
    return path, util.run_engine(oracle, path, prompts(), **PASSES)["steps"]


@pytest.mark.gpu
@pytest.mark.parametrize("height,kv_bytes", [(4, 4), (6, 2), (9, 4), (9, 2)])
def test_passes_through_every_epilogue(passes, tmp_path, height, kv_bytes):
    path, want = passes
    dst = str(tmp_path / "got.npz")
    env = dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_GEMM_WIDE=str(height))
    r = subprocess.run([sys.executable, "-c", CHILD, path, dst, str(kv_bytes)], env=env, capture_output=True, text=True, timeout=150)
    assert r.returncode == 0, r.stderr[-2000:]
    got = np.load(dst)
    for i, o in enumerate(want):
        np.testing.assert_array_equal(got[f"sampled{i}"], o["sampled"])
        assert np.abs(got[f"logits{i}"] - o["logits"]).max() < (2e-4 if kv_bytes == 4 else 2e-3)   # the bars of the forward pass


BF16_CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import hybrid_util, test_gpu_wide
eng = hybrid_util.engine(capi.load_hip(), sys.argv[1], False, tokens=704)
got = hybrid_util.feed_all(eng, [[(0, 300), (1, 257)], [(0, 133)]], test_gpu_wide.bf16_sequences())
eng.close()
np.savez(sys.argv[2], **{str(q): rows for q, rows in got.items()})
"""


def bf16_sequences():
    return {0: hybrid_util.tokens(433, 203, 1), 1: hybrid_util.tokens(257, 203, 2)}


@pytest.fixture(scope="module")
def bf16_passes(tmp_path_factory):
    # K of 9 and 13 steps; dense, gated and row projections whose widths end inside a tile of 256 features
    cfg = synth.hybrid_config(288, 203, [(hybrid_util.A(6, 2, 48, 64, size=150, keep_first=3, taps=3, rot=16), hybrid_util.E(64, 4, 2, 416)),
                                         (hybrid_util.L(3, 64, 64), 800)])
    path, cfg, w = hybrid_util.model(tmp_path_factory.mktemp("wide_bf16"), "wide", cfg=cfg)
    return path, {q: hybrid_oracle.forward(cfg, w, seq) for q, seq in bf16_sequences().items()}


@pytest.mark.gpu
@pytest.mark.parametrize("height", [4, 6, 8, 10])
def test_bf16_passes(bf16_passes, tmp_path, height):
    path, want = bf16_passes
    dst = str(tmp_path / "got.npz")
    env = dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_GEMM_WIDE=str(height))
    r = subprocess.run([sys.executable, "-c", BF16_CHILD, path, dst], env=env, capture_output=True, text=True, timeout=150)
    assert r.returncode == 0, r.stderr[-2000:]
    got = np.load(dst)
    for q, o in want.items():
        assert hybrid_util.error(got[str(q)], o) < hybrid_util.limit(False), q   # the bar of the design's whole passes


RULE_CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import hybrid_util, test_gpu_row_scale, test_gpu_wide
lib = capi.load_hip()
if sys.argv[3] == "f16":
    lib.init_ops()
    rows = test_gpu_row_scale.logits(lib, sys.argv[1], test_gpu_wide.RULE_TOKENS)
else:
    eng = hybrid_util.engine(lib, sys.argv[1], False, tokens=704)
    rows = hybrid_util.feed_all(eng, [[(0, test_gpu_wide.RULE_TOKENS)]], {0: test_gpu_wide.rule_tokens()})[0]
    eng.close()
np.save(sys.argv[2], rows)
"""
RULE_TOKENS = 700


def rule_tokens():
    return np.arange(RULE_TOKENS, dtype=np.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["f16", "bf16"])
def test_the_launchers_own_rules(oracle, tmp_path, kind):
    """Gated pairs of 2,816 x 1,024 at 700 tokens: 242 tiles of 256 x 64 for 256 CUs, K of 32 steps, which both rules take.  The
    smaller tiles add the same products in the same order: the same bits."""
    path = str(tmp_path / "model")
    if kind == "f16":
        synth.write_model(path, synth.ModelShape(dim=1024, hidden_dim=2816, n_layers=1, n_heads=16, n_kv_heads=4, vocab_size=RULE_TOKENS, max_seq_len=704), seed=4)
        want = test_gpu_row_scale.logits(oracle, path, RULE_TOKENS)
    else:
        cfg = synth.latent_config(1024, RULE_TOKENS, [(synth.latent_mixer(4, 32, 16, 32, 64, 64), 2816)])
        want = latent_oracle.forward(cfg, latent_util.model(tmp_path, "rule", cfg=cfg)[2], rule_tokens())
        path = str(tmp_path / "rule_3")
    got = []
    for env in ({}, {"NVLLM_GEMM_WIDE": "0"}):
        dst = str(tmp_path / f"got{len(got)}.npy")
        r = subprocess.run([sys.executable, "-c", RULE_CHILD, path, dst, kind], capture_output=True, text=True, timeout=150,
                           env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), **env))
        assert r.returncode == 0, r.stderr[-2000:]
        got.append(np.load(dst))
    np.testing.assert_array_equal(got[0], got[1])
    if kind == "f16":
        assert np.abs(got[0] - want).max() < 2e-4   # the bar of the forward pass
    else:
        assert hybrid_util.error(got[0], want) < hybrid_util.limit(False)
