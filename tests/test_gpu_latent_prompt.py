"""Prompt portions of the Suselorn design with keys and values formed from the cached latents (csrc/latent_prompt.hip), against the
attention over latents that single tokens take: the same tokens as one prompt, in portions that end inside pages, pairs and
blocks of keys, beside single tokens, on blocks of one and of four pages, and at head sizes of every form.  Which way portions go is read
from the environment once per process, hence a child process each."""
import os
import subprocess
import sys

import numpy as np
import pytest

from nvllm_amd import synth
from tests import latent_oracle as O
from tests import latent_util as U
from tests.test_gpu_latent_order import flops_of

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
M = synth.latent_mixer
CONFIGS = dict(U.CONFIGS,
               # every width of unrotated, rotated and value parts that has a form, and one (96) that has none
               sizes=synth.latent_config(64, 130, [(M(2, 128, 64, 128, 96, 32), 40), (M(9, 30, 20, 60, 512, 32), None), (M(3, 64, 32, 32, 40, 32), 48),
                                                   (M(8, 64, 64, 64, 256, 32), None), (M(2, 96, 32, 32, 64, 32), 40)], streams=2))
LENGTHS = {0: 333, 1: 150, 2: 40, 3: 97}
PLANS = {
    "prompts": [[(0, 333), (1, 150)], [(2, 40), (3, 97)]],
    "portions": [[(0, 130), (1, 17)], [(0, 65), (1, 33), (2, 5)], [(0, 64), (1, 49), (2, 2)], [(0, 74), (1, 51), (2, 33)], [(3, 97)]],
    # single tokens before, between and behind portions
    "mixed": [[(0, 100), (1, 20)], [(1, 1), (0, 33), (2, 1), (3, 50)], [(0, 16), (2, 1), (1, 128), (3, 1)], [(3, 45), (0, 183), (2, 1)], [(2, 37), (3, 1), (0, 1), (1, 1)]],
}
CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import latent_util as U, test_gpu_latent_prompt as me
lib = capi.load_hip()
out = {}
for block_size in (16, 64):
    for what, plan in me.PLANS.items():
        eng = U.engine(lib, sys.argv[1], False, tokens=1024, block_size=block_size)
        got = U.feed_all(eng, plan, me.sequences(int(sys.argv[3])))
        eng.close()
        out.update({"%s %d %d" % (what, block_size, q): rows for q, rows in got.items()})
np.savez(sys.argv[2], **out)
"""


def sequences(vocab):
    return {q: U.tokens(n, vocab, 40 + q) for q, n in LENGTHS.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_portions_agree_with_attention_over_latents(tmp_path, name):
    path, cfg, w = U.model(tmp_path, name, seed=5, cfg=CONFIGS[name])
    seqs = sequences(cfg["vocab"])
    want = {q: O.forward(cfg, w, seq) for q, seq in seqs.items()}
    error = []
    for way in ("0", "1"):
        dst = str(tmp_path / (way + ".npz"))
        r = subprocess.run([sys.executable, "-c", CHILD, path, dst, str(cfg["vocab"])], capture_output=True, text=True, timeout=150,
                           env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_LATENT_EXPAND=way))
        assert r.returncode == 0, r.stderr[-2000:]
        got = np.load(dst)
        assert len(got.files) == 2 * sum(len({q for step in p for q, _ in step}) for p in PLANS.values())
        square = lambda rows: float((rows * rows).sum())  # noqa: E731
        off, size = 0.0, 0.0
        for k in got.files:
            o = want[int(k.split()[-1])][:len(got[k])]
            d = got[k].astype(np.float64) - o
            off, size = off + square(d - d.mean(-1, keepdims=True)), size + square(o)
        error.append((off / size) ** 0.5)
    # Both ways round as often, keys instead of absorbed queries and values instead of attended latents: the same error, in which
    # runs of a few hundred rows scatter by a tenth (0.86 to 1.12 over 36 models).
    assert error[1] < 1.25 * error[0] and error[1] < U.limit(False) / 2, error


@pytest.mark.gpu
@pytest.mark.parametrize("heads,rank,length,formings", [(32, 512, 600, 4), (24, 256, 600, 4), (17, 100, 1300, 2), (32, 480, 600, 8), (16, 512, 600, 8)])
def test_forming_beside_tokens_that_come_alone(hip, tmp_path, heads, rank, length, formings):
    """Items of 32 columns (17 to 32 heads) of the widest row and of one with up to eight tiles share a launch with the forming of keys and values; others
    do not.  One, three and twenty such tokens (few and, for the last pass's portion, too many workgroups) beside long portions."""
    cfg = synth.latent_config(64, 130, [(M(heads, 64, 64, 64, rank, 32), 40)] * 2, streams=2)
    path, cfg, w = U.model(tmp_path, "beside", seed=heads, cfg=cfg)
    n = 22
    seqs = {q: U.tokens(length + 190 if q == 0 else length if q == 1 else 40, 130, 70 + q) for q in range(n)}
    plan = [[(q, 30) for q in range(2, n)], [(0, length), (5, 1)], [(3, 1), (1, length), (4, 1), (6, 1)], [(q, 1) for q in range(2, 12)] + [(0, 190)] + [(q, 1) for q in range(12, n)]]
    eng = U.engine(hip, path, False, slots=n, tokens=4096)
    hip.nvllm_prof_reset()
    hip.nvllm_prof_enable(1)
    try:
        got = U.feed_all(eng, plan, seqs)
    finally:
        hip.nvllm_prof_enable(0)
    assert flops_of(hip, "latent_expand")[0] == formings   # launches of its own, two layers a pass: the first has no single tokens
    hip.nvllm_prof_reset()
    eng.close()
    for q, rows in got.items():
        assert U.error(rows, O.forward(cfg, w, seqs[q][:len(rows)])) < U.limit(False), q
