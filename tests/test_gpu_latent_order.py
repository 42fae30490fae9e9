"""Single tokens before, between and behind prompt portions that form their keys and values (csrc/latent_prompt.hip): the same bits
wherever the scheduler puts them, and as few tokens through the products of the attention over latents."""
import ctypes as C

import numpy as np
import pytest

from nvllm_amd import synth
from tests import latent_util as U

pytestmark = pytest.mark.gpu
CONFIG = synth.latent_config(64, 130, [(synth.latent_mixer(8, 64, 32, 64, 512, 48), 40)] * 2, streams=2)
PROMPTS, ROWS, LONG = (0, 1), (2, 3, 4), 640
ORDERS = {"behind": [0, 1, 2, 3, 4], "before": [2, 3, 4, 0, 1], "between": [0, 2, 3, 1, 4], "around": [2, 0, 3, 1, 4], "ends": [3, 0, 1, 4, 2]}


def flops_of(hip, name):
    for c in range(hip.nvllm_prof_num_classes()):
        n, ms, by, fl = C.c_longlong(), C.c_double(), C.c_double(), C.c_double()
        hip.nvllm_prof_get(c, C.byref(n), C.byref(ms), C.byref(by), C.byref(fl))
        if hip.nvllm_prof_name(c).decode() == name:
            return n.value, fl.value


def test_any_order(hip, tmp_path):
    path, cfg, _ = U.model(tmp_path, "order", seed=5, cfg=CONFIG)
    seqs = {q: U.tokens(LONG + 4 if q in PROMPTS else 70 + 9 * q, 130, q) for q in PROMPTS + ROWS}
    got, figures = {}, {}
    for name, order in ORDERS.items():
        eng = U.engine(hip, path, False, slots=5, tokens=2048)
        hip.nvllm_prof_reset()
        try:
            for q in ROWS:
                eng.feed(q, seqs[q][:-2], [0])
            eng.feed_run()
            out = {q: [] for q in seqs}
            hip.nvllm_prof_enable(1)
            for step in range(2):   # the second time portions of four tokens, which attend over the latents
                for q in order:
                    at = (0 if q in PROMPTS else len(seqs[q]) - 2) + (step if q in ROWS else LONG * step)
                    n = 1 if q in ROWS else (LONG, 4)[step]
                    eng.feed(q, seqs[q][at:at + n], range(n))
                rows = eng.feed_run()
                i = 0
                for q in order:
                    n = 1 if q in ROWS else (LONG, 4)[step]
                    out[q].append(rows[i:i + n])
                    i += n
            hip.nvllm_prof_enable(0)
            figures[name] = [flops_of(hip, c) for c in ("gemm_absorb", "latent_expand")]
            got[name] = {q: np.concatenate(r) for q, r in out.items()}
        finally:
            hip.nvllm_prof_enable(0)
            hip.nvllm_prof_reset()
            eng.close()
    for name in ORDERS:
        assert figures[name] == figures["behind"], name
        for q in seqs:
            np.testing.assert_array_equal(got[name][q], got["behind"][q], err_msg="%s %d" % (name, q))
    assert figures["behind"][1][0] == 2
