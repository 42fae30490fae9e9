"""Tokens whose attention over the latents is cut into slices: merged and multiplied by W_uv in one launch.  Batches at the edges of eight
and sixteen tokens and of the launch's limit, two to many slices, portions beside single tokens, rows and heads of every width it takes."""
import numpy as np
import pytest

from nvllm_amd import synth
from tests import latent_oracle as O
from tests import latent_util as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,vdim,rank", [(3, 32, 64), (2, 128, 512), (5, 40, 160), (33, 20, 40)])
def test_sliced_tokens_through_their_value_products(hip, tmp_path, heads, vdim, rank):
    cfg = synth.latent_config(64, 131, [(synth.latent_mixer(heads, 32, 16, vdim, rank, 48), 64)] * 2, streams=2)
    path, cfg, weights = U.model(tmp_path, "value", seed=heads, cfg=cfg)
    slots = 18
    eng = U.engine(hip, path, False, slots=slots, tokens=slots * 320)
    for rows, portion in ((1, 0), (8, 3), (9, 0), (17, 5)):
        lengths = {r: 300 - 13 * r for r in range(rows)}
        seqs = {r: U.tokens(n, 131, 7 * r + rows) for r, n in lengths.items()}
        plan = [[(r, n - 1)] for r, n in lengths.items()]
        last = [(r, 1) for r in seqs]
        if portion:   # a short portion in the same pass
            seqs[rows] = U.tokens(280, 131, 99)
            plan.append([(rows, 280 - portion)])
            last.append((rows, portion))
        got = U.feed_all(eng, plan + [last], seqs)
        for r, seq in seqs.items():
            assert U.error(got[r], O.forward(cfg, weights, seq)) < U.limit(False), (rows, r)
    eng.close()
