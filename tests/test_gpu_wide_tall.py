"""The 256-feature tiles (csrc/gemm_wide.h) of bf16 models at the heights that eight waves share, and of five blocks, with the query
projection among them: whole passes at a height read from the environment, widths and token counts that end inside a tile."""
import numpy as np
import pytest

from nvllm_amd import synth
from tests import hybrid_oracle, hybrid_util, latent_oracle, latent_util, test_gpu_waves

# K of 9 and 13 steps, and of 9 in the query projection
CONFIGS = {"hybrid": (test_gpu_waves.HYBRID, hybrid_util, hybrid_oracle),
           "latent": (synth.latent_config(288, 203, [(synth.latent_mixer(5, 32, 32, 48, 160, 288), 416)] * 2, streams=2), latent_util, latent_oracle)}


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    out = {}
    for kind, (cfg, util, oracle) in CONFIGS.items():
        path, cfg, w = util.model(tmp_path_factory.mktemp("tall_" + kind), kind, cfg=cfg)
        out[kind] = path, {q: oracle.forward(cfg, w, seq) for q, seq in test_gpu_waves.sequences().items()}
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("height", [5, 8, 10, 12, 14, 16])
@pytest.mark.parametrize("kind", sorted(CONFIGS))
def test_bf16_passes(folders, tmp_path, kind, height):
    path, want = folders[kind]
    dst = str(tmp_path / "got.npz")
    test_gpu_waves.child(test_gpu_waves.FOLDER_CHILD, path, dst, kind, NVLLM_GEMM_WIDE=str(height))
    got = np.load(dst)
    for q, o in want.items():
        assert hybrid_util.error(got[str(q)], o) < hybrid_util.limit(False), q   # the bar of the designs' whole passes
