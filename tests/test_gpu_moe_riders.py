"""Passes of few tokens, whose router and choice of experts ride on the shared expert's products: at the edges of a token block, of the
chosen tile heights and of the passes that launch them apart; routers of one and of several feature tiles."""
import os
import subprocess
import sys

import numpy as np
import pytest

from nvllm_amd import synth
from tests import hybrid_oracle as O
from tests import hybrid_util as U
from tests.test_gpu_latent_order import flops_of

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


def passes(hip, path, tokens):
    """Logits of a prompt per count, and the launches of a router and of a choice apart in them."""
    eng = U.engine(hip, path, False, slots=1, tokens=2208)
    out = {}
    hip.nvllm_prof_reset()
    hip.nvllm_prof_enable(1)
    try:
        for n in tokens:
            out[str(n)] = U.feed_all(eng, [[(0, n)]], {0: U.tokens(n, 211, n)})[0]
    finally:
        hip.nvllm_prof_enable(0)
    out["apart"] = np.array([flops_of(hip, c)[0] for c in ("gemm_router", "route")])
    hip.nvllm_prof_reset()
    eng.close()
    return out


CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import test_gpu_moe_riders
np.savez(sys.argv[2], **test_gpu_moe_riders.passes(capi.load_hip(), sys.argv[1], [int(n) for n in sys.argv[3:]]))
"""


# Tiles: the launchers' own; K dealt to four waves (one height of 22 x 11 tiles, which leave fewer CUs than there are groups of token blocks, so
# that a rider has two); 256 features by four waves (19 x 13) and by eight (35 x 7), the same.  Squares in 9, 35 and 65 sums, two of them past the parts
# (32; 16 of 2,100 tokens with four row blocks).  200 tokens: the first product in tiles, the second streaming.  Eight experts a token: apart, as one wave's
# choices for 16 tokens would outlast the tiles
@pytest.mark.parametrize("env,width,shared,experts,top,tokens", [
    ({}, 288, 96, 31, 3, (256, 257, 1100)), ({}, 288, 96, 63, 2, (511, 2100)), ({}, 1100, 96, 15, 2, (300,)), ({}, 2080, 64, 63, 2, (256, 2100)), ({}, 288, 2816, 16, 2, (200,)),
    ({"NVLLM_GEMM_WAVES": "6"}, 1024, 1408, 16, 2, (1029,)), ({"NVLLM_GEMM_WAVES": "2"}, 1100, 416, 40, 2, (433,)),
    ({"NVLLM_GEMM_WIDE": "4"}, 1024, 2400, 31, 2, (800,)), ({"NVLLM_GEMM_WIDE": "8"}, 512, 4480, 5, 2, (800,)), ({"NVLLM_GEMM_WIDE": "12"}, 1100, 416, 63, 2, (433,)),
    ({}, 288, 96, 63, 8, (400,))])
def test_the_same_choices_as_apart(hip, tmp_path, env, width, shared, experts, top, tokens):
    """A shared expert whose second matrix is zero against none at all: only who forms logits and choices differs, and no bit may."""
    window = synth.window_mixer(4, 2, 16, 16, size=48, keep_first=4)
    got = []
    for ff in (shared, None):
        cfg = synth.hybrid_config(width, 211, [(window, synth.expert_mlp(48, experts, top, ff))] * 2)
        if ff:
            path, _, weights = U.model(tmp_path, "rides", seed=experts, cfg=cfg, edit=lambda name, v: 0 * v if name.endswith("shared.down") else None)
        else:
            path, _, _ = U.model(tmp_path, "apart", seed=experts, cfg=cfg, edit=lambda name, v: weights[name])
        if env:
            dst = str(tmp_path / ("got%d.npz" % len(got)))
            r = subprocess.run([sys.executable, "-c", CHILD, path, dst, *map(str, tokens)], capture_output=True, text=True, timeout=110,
                               env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), **env))
            assert r.returncode == 0, r.stderr[-2000:]
            got.append(np.load(dst))
        else:
            got.append(passes(hip, path, tokens))
    assert got[0]["apart"][0] == (2 if top == 8 else 0) and got[1]["apart"][0] == 2 * len(tokens)
    for n in tokens:
        np.testing.assert_array_equal(got[0][str(n)], got[1][str(n)], err_msg=str(n))


@pytest.mark.parametrize("f32,shared", [(True, 8), (True, None), (False, 8)])
def test_more_experts_than_the_limit_are_refused(tmp_path, monkeypatch, f32, shared):
    """4,096 experts, whoever chooses among them: refused before the pass launches anything."""
    cfg = synth.hybrid_config(32, 64, [(synth.window_mixer(1, 1, 8, 8, size=16, keep_first=1), synth.expert_mlp(4, 4097, 2, shared))])
    monkeypatch.setattr(synth, "_tensor_values", lambda shape, kind, rng, routed: rng.standard_normal(shape))
    path, _, _ = U.model(tmp_path, "many", cfg=cfg)
    code = ("import sys\nfrom nvllm_amd import capi\nfrom tests import hybrid_util as U\neng = U.engine(capi.load_hip(), sys.argv[1], %r, slots=1, tokens=64)\n"
            "eng.feed(0, [1, 2, 3], range(3))\neng.feed_run()\nprint('survived')\n" % f32)
    r = subprocess.run([sys.executable, "-c", code, path], capture_output=True, text=True, timeout=110,
                       env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", "")))
    assert r.returncode != 0 and "survived" not in r.stdout
    assert "2 of 4097 experts" in r.stderr, r.stderr[-500:]


@pytest.mark.parametrize("f32", [True, False], ids=["fp32", "bf16"])
@pytest.mark.parametrize("experts,top,rides,apart", [(16, 2, (8, 64, 80), ()), (64, 8, (16,), (192,)), (128, 2, (16,), (96, 128)), (128, 8, (), (64, 128))])
def test_long_choices_are_launched_apart(hip, tmp_path, f32, experts, top, rides, apart):
    """One workgroup beside a product's tiles chooses only where it is about as soon done as a launch of its own (route_rides); who chooses shows in no bit."""
    if not f32:
        rides, apart = [n for n in rides if n <= 128], [n for n in apart if n <= 128]   # (more tokens take tiles, which carry other riders)
    window = synth.window_mixer(4, 2, 16, 16, size=48, keep_first=4)
    cfg = synth.hybrid_config(128, 211, [(window, synth.expert_mlp(16, experts, top, 256))])
    path, cfg, weights = U.model(tmp_path, "long", seed=experts, cfg=cfg)
    eng = U.engine(hip, path, f32, slots=1)
    try:
        for n in sorted([*rides, *apart]):
            seq = U.tokens(n, 211, n)
            hip.nvllm_prof_reset()
            hip.nvllm_prof_enable(1)
            got = U.feed_all(eng, [[(0, n)]], {0: seq})[0]
            hip.nvllm_prof_enable(0)
            assert flops_of(hip, "route")[0] == (n in apart), n
            assert U.error(got, O.forward(cfg, weights, seq)) < U.limit(f32), n
    finally:
        hip.nvllm_prof_enable(0)
        hip.nvllm_prof_reset()
        eng.close()
