"""Experts whose rows are sorted into groups as tall as a 256-feature tile (csrc/gemm_wide_b16.hip, expert_rows_wide), at every height:
widths that end inside a tile, an expert without rows, one with more than a group's, groups that are no power of two.  The
height is read from the environment once per process, hence a child process per height."""
import os
import subprocess
import sys

import numpy as np
import pytest

from tests import hybrid_oracle as O
from tests.test_gpu_latent_ops import rng, rounded
from tests.test_gpu_waves import ROOT

HEIGHTS = (4, 5, 6, 8, 10, 12, 14, 16)
# tokens, width, hidden width, experts, choices: K of 9 and 10 steps, N of 640 and 288; of 8 and 9, N of 576 and 256; one expert for all
SHAPES = [(300, 288, 320, 5, 2), (150, 256, 288, 9, 3), (270, 320, 256, 1, 1)]
CHILD = """
import sys
import numpy as np
from nvllm_amd import capi
from tests import test_gpu_experts_wide as me
from tests.test_gpu_latent_ops import Dev
hip = capi.load_hip()
hip.init_ops()
out = {}
for i, shape in enumerate(me.SHAPES):
    T, D, ff, E, top = shape
    x, z, gate, up, down = me.case(shape)
    d = Dev(hip)
    y, choice = d.empty(T * D), d.empty(T * top)
    hip.nvllm_expert_ff(y, choice, None, d(x), d(z), d(gate), d(up), d(down), D, ff, E, top, 2, T)
    out["y%d" % i], out["choice%d" % i] = hip.to_host(y, (T, D)), hip.to_host(choice, (T, top), np.int32)
    d.close()
np.savez(sys.argv[1], **out)
"""


def case(shape):
    T, D, ff, E, top = shape
    r = rng(T + E)
    z = r.permuted(np.tile(np.linspace(-2.5, 2.0, E), (T, 1)), axis=1)
    if E > 2:
        z[:, 1] = 3.0      # everybody's
        z[:, 3] = -4.0     # nobody's
    weights = [rounded(r.standard_normal(s) * s[-1] ** -0.5, 2) for s in ((E, ff, D), (E, ff, D), (E, D, ff))]
    return [rounded(r.standard_normal((T, D)), 2), z, *weights]


def wanted(shape):
    T, D, ff, E, top = shape
    x, z, gate, up, down = case(shape)
    chosen, weight = O.route(z, top)
    want = np.zeros((T, D))
    for e in range(E):
        t, j = np.nonzero(chosen == e)
        if len(t):
            want[t] += O.gated(weight[t, j][:, None] * x[t], gate[e], up[e], down[e])
    return chosen, want


@pytest.fixture(scope="module")
def wants():
    return [wanted(s) for s in SHAPES]


@pytest.mark.gpu
@pytest.mark.parametrize("height", HEIGHTS)
def test_every_height(wants, tmp_path, height):
    dst = str(tmp_path / "got.npz")
    r = subprocess.run([sys.executable, "-c", CHILD, dst], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""), NVLLM_GEMM_WIDE=str(height)))
    assert r.returncode == 0, r.stderr[-2000:]
    got = np.load(dst)
    for i, (chosen, want) in enumerate(wants):
        np.testing.assert_array_equal(got["choice%d" % i], chosen)
        assert np.abs(got["y%d" % i] - want).max() < 1e-2 * np.abs(want).max(), SHAPES[i]   # the bar of test_gpu_hybrid_ops.py


# sixteen (eight) experts of 2 x ff x width, rows of a batch of T tokens with two choices: those that measured slower in these tiles stay out
@pytest.mark.gpu
@pytest.mark.skipif("NVLLM_GEMM_WIDE" in os.environ, reason="the environment forces a height")
@pytest.mark.parametrize("width,ff,experts,T,height", [
    (1792, 1024, 16, 512, 0), (1792, 1024, 16, 640, 0), (1792, 1024, 16, 800, 8), (1664, 832, 16, 800, 0),      # 50 and 44 % of 256 CUs; K of 832
    (2048, 1152, 16, 400, 0), (2304, 1152, 16, 400, 0), (2048, 1152, 16, 512, 6), (2304, 1152, 16, 512, 6),     # 56 %
    (3328, 1664, 8, 330, 0), (3328, 1664, 8, 512, 10),                                                          # 41 %
    (1792, 1280, 16, 330, 4), (2048, 1280, 16, 330, 4), (2560, 1280, 16, 400, 5), (2048, 1408, 16, 1029, 10),   # 62, 62, 62, 69 %
    (1536, 1280, 16, 800, 0), (2048, 1408, 16, 300, 0), (2048, 1408, 16, 2000, 0)])                             # 37 % of the second; few rows; many
def test_which_batches_take_them(hip, width, ff, experts, T, height):
    assert hip.dll.nvllm_internal_expert_rows_wide(2 * T, experts, 2 * ff, width, width, ff) == 16 * height
