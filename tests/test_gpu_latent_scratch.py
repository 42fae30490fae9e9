"""Prompt portions of the Suselorn design whose keys and values (csrc/latent_prompt.hip) find no memory: a limit on their bytes stands
for an allocation that fails, in every layer or in the one with more heads.  Those layers attend over the latents."""
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
CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import latent_util as U
eng = U.engine(capi.load_hip(), sys.argv[1], False, tokens=1024)
out = U.feed_all(eng, [[(0, 100), (1, 20)], [(1, 1), (0, 33)], [(0, 12), (1, 60)]], {0: U.tokens(145, 130, 1), 1: U.tokens(81, 130, 2)})
eng.close()
np.savez(sys.argv[2], *(out[q] for q in (0, 1)))
"""


def test_layers_without_memory(tmp_path):
    cfg = synth.latent_config(64, 130, [(synth.latent_mixer(8, 64, 32, 64, 64, 32), 40), (synth.latent_mixer(2, 64, 32, 64, 64, 32), 40)], streams=2)
    path, cfg, w = U.model(tmp_path, "scratch", seed=5, cfg=cfg)
    want = [O.forward(cfg, w, U.tokens(n, 130, q)) for n, q in ((145, 1), (81, 2))]

    def rows(way, most):
        dst = str(tmp_path / "rows.npz")
        r = subprocess.run([sys.executable, "-c", CHILD, path, dst], capture_output=True, text=True, timeout=100,
                           env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_LATENT_EXPAND=way,
                                    NVLLM_LATENT_EXPAND_BYTES=str(most)))
        assert r.returncode == 0, r.stderr[-2000:]
        got = np.load(dst)
        got = [got[k] for k in got.files]
        for g, o in zip(got, want):
            assert U.error(g, o) < U.limit(False), (way, most)
        return np.concatenate(got)

    over_latents, formed = rows("0", 1e9), rows("1", 1e9)
    np.testing.assert_array_equal(rows("1", 0), over_latents)
    one = rows("1", 8 * 2 * 32 * 2 * 128)   # eight pairs of pages, two heads: all passes of those; none of the five pairs and more with eight heads
    assert (one != over_latents).any() and (one != formed).any()
