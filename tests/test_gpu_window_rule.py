"""Which single tokens' windows are cut into slices: for every form of the kernel, lengths on both sides of the line."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_hybrid_ops import filled, reference
from tests.test_gpu_latent_ops import rng, rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,vdim,length,sliced", [(64, 64, 1536, False), (64, 64, 1537, True), (48, 32, 1500, False), (128, 128, 960, False), (128, 128, 961, True),
                                                    (96, 64, 1100, True), (256, 256, 576, False), (256, 256, 577, True), (192, 192, 320, False), (192, 192, 321, True),
                                                    (160, 256, 400, True)])
def test_slices(hip, dim, vdim, length, sliced):
    pool, kv = filled(hip, 2, dim, vdim, 2, 16, [length, 5], dim)
    q = rounded(rng(length).standard_normal((2, 8, dim)), 2)
    hip.nvllm_prof_reset()
    hip.nvllm_prof_enable(1)
    try:
        got = pool.attend([0, 1], [length - 1, 4], q, dim ** -0.5, 20.0, 1 << 30, 4)
    finally:
        hip.nvllm_prof_enable(0)
    merges = 0
    for c in range(hip.nvllm_prof_num_classes()):
        n, ms, by, fl = C.c_longlong(), C.c_double(), C.c_double(), C.c_double()
        hip.nvllm_prof_get(c, C.byref(n), C.byref(ms), C.byref(by), C.byref(fl))
        if hip.nvllm_prof_name(c) == b"attn_combine":
            merges = n.value
    hip.nvllm_prof_reset()
    want = reference(kv, q, [length - 1, 4], [0, 1], dim ** -0.5, 20.0, 1 << 30, 4)
    pool.close()
    assert np.abs(got - want).max() < 1.2e-2 * np.abs(want).max()   # the bar of test_gpu_hybrid_ops.py
    assert merges == int(sliced)
