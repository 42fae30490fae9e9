"""The bytes and operations that the kernel timing reports for the experts' products of fp32 rows: those of the pairs of a token
and a choice and of the experts they can reach, not of the padding the launch has room for."""
import ctypes as C

import pytest

from tests.test_gpu_latent_ops import Dev, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,D,ff,E,top", [(1, 64, 32, 16, 2), (3, 64, 48, 16, 2), (80, 64, 32, 16, 2), (40, 63, 21, 3, 1)])
def test_experts_of_fp32_rows(hip, T, D, ff, E, top):
    r, d = rng(T), Dev(hip)
    args = [d(r.standard_normal(s)) for s in ((T, D), (T, E), (E, ff, D), (E, ff, D), (E, D, ff))]
    out = d.empty(T * D)
    hip.nvllm_prof_reset()
    hip.nvllm_prof_enable(1)
    try:
        hip.nvllm_expert_ff(out, None, None, *args, D, ff, E, top, 4, T)
    finally:
        hip.nvllm_prof_enable(0)
    got = {}
    for c in range(hip.nvllm_prof_num_classes()):
        n, ms, by, fl = C.c_longlong(), C.c_double(), C.c_double(), C.c_double()
        hip.nvllm_prof_get(c, C.byref(n), C.byref(ms), C.byref(by), C.byref(fl))
        if n.value:
            got[hip.nvllm_prof_name(c).decode()] = (n.value, by.value, fl.value)
    hip.nvllm_prof_reset()
    d.close()
    pairs = T * top
    touched = min(E, pairs)
    assert got["gemm_expert_up"] == (1, 4.0 * (touched * 2 * ff * D + pairs * (D + ff)), 2.0 * pairs * 2 * ff * D)
    assert got["gemm_expert_down"] == (1, 4.0 * (touched * D * ff + pairs * (ff + D)), 2.0 * pairs * D * ff)
