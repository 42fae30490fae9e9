"""Passes of few tokens, whose router and choice of experts ride on the shared expert's products: at the edges of a token block, of the
chosen tile heights and of the passes that launch them apart; routers of one and of several feature tiles."""
import numpy as np
import pytest

from nvllm_amd import synth
from tests import hybrid_oracle as O
from tests import hybrid_util as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,shared", [(5, 40), (40, 96), (70, 64)])
def test_passes_of_few_tokens(hip, tmp_path, experts, shared):
    window = synth.window_mixer(4, 2, 16, 16, size=48, keep_first=4)
    cfg = synth.hybrid_config(128, 211, [(window, synth.expert_mlp(48, experts, 2, shared)), (window, synth.expert_mlp(48, experts, 2, shared))])
    path, cfg, weights = U.model(tmp_path, "riders", seed=experts, cfg=cfg)
    eng = U.engine(hip, path, False, slots=1)
    for n in (1, 16, 17, 64, 65, 255, 256):
        seq = U.tokens(n, 211, n)
        got = U.feed_all(eng, [[(0, n)]], {0: seq})[0]
        assert U.error(got, O.forward(cfg, weights, seq)) < U.limit(False), n
    eng.close()


# routers of one row block, of two and of four, and one wider than rides; 256 tokens and more take tiles whose idle CUs carry them
@pytest.mark.parametrize("experts,top", [(5, 2), (31, 3), (63, 4), (64, 2)])
def test_prompts(hip, tmp_path, experts, top):
    window = synth.window_mixer(4, 2, 16, 16, size=48, keep_first=4)
    cfg = synth.hybrid_config(288, 211, [(window, synth.expert_mlp(48, experts, top, 96))] * 2)
    path, cfg, weights = U.model(tmp_path, "prompts", seed=experts, cfg=cfg)
    eng = U.engine(hip, path, False, slots=1)
    for n in (256, 257, 511, 1100):
        seq = U.tokens(n, 211, n)
        got = U.feed_all(eng, [[(0, n)]], {0: seq})[0]
        np.testing.assert_array_equal(U.feed_all(eng, [[(0, n)]], {0: seq})[0], got)
        assert U.error(got, O.forward(cfg, weights, seq)) < U.limit(False), n
    eng.close()


# in 32 bits the choice rides on the shared expert's first product up to 256 tokens; without a shared expert, and with rows that are no multiples of 16 bytes, nobody rides
@pytest.mark.parametrize("width,experts,shared", [(128, 5, 40), (96, 70, 96), (64, 16, None), (66, 6, 48)])
def test_choices_in_32_bits(hip, tmp_path, width, experts, shared):
    window = synth.window_mixer(4, 2, 16, 16, size=48, keep_first=4)
    cfg = synth.hybrid_config(width, 211, [(window, synth.expert_mlp(48, experts, 2, shared))] * 2)
    path, cfg, weights = U.model(tmp_path, "choices", seed=experts, cfg=cfg)
    eng = U.engine(hip, path, True, slots=1)
    for n in (1, 17, 128, 129, 256, 257):
        seq = U.tokens(n, 211, n)
        got = U.feed_all(eng, [[(0, n)]], {0: seq})[0]
        np.testing.assert_array_equal(U.feed_all(eng, [[(0, n)]], {0: seq})[0], got)
        assert U.error(got, O.forward(cfg, weights, seq)) < U.limit(True), n
    eng.close()


# K splits of both products; of the second, with 96-feature tiles of the first from 33 tokens on
@pytest.mark.parametrize("width,experts,shared", [(1024, 20, 96), (512, 70, 2816), (256, 30, 2816)])
def test_riders_beside_k_splits(hip, tmp_path, width, experts, shared):
    """The same bits twice: riders share the launch, and the CUs, with tiles whose partial sums meet through memory."""
    window = synth.window_mixer(4, 2, 16, 16, size=48, keep_first=4)
    cfg = synth.hybrid_config(width, 211, [(window, synth.expert_mlp(48, experts, 2, shared))] * 2)
    path, cfg, weights = U.model(tmp_path, "splits", seed=experts, cfg=cfg)
    eng = U.engine(hip, path, False, slots=1)
    for n in (1, 16, 40, 64, 65, 128, 200):
        seq = U.tokens(n, 211, n)
        got = U.feed_all(eng, [[(0, n)]], {0: seq})[0]
        np.testing.assert_array_equal(U.feed_all(eng, [[(0, n)]], {0: seq})[0], got)
        assert U.error(got, O.forward(cfg, weights, seq)) < U.limit(False), n
    eng.close()
