"""Logits rows of a pass that is waited for: the classifier stores them into RunState.logits itself, where that is the page-locked
array of malloc_run_state; any other memory, and a pass sent ahead, is served by a copy.  Same bits every way."""
import ctypes as C

import numpy as np
import pytest

from nvllm_amd import capi
from tests import latent_util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["fp16", "fp32", "odd-bf16", "odd-f32"])   # (the odd ones: 203 words, capped logits)
def test_rows_are_the_same_every_way(hip, tmp_models, tmp_path, kind):
    f32 = kind.endswith("f32")
    hip.nvllm_set_compute_dtype(capi.COMPUTE_F32 if f32 else capi.COMPUTE_BF16)
    folder = kind.startswith("odd")
    path = latent_util.model(tmp_path, "odd")[0] if folder else tmp_models("tiny", dtype="f32", exact16=False)[0] if kind == "fp32" else tmp_models("tiny")[0]
    w, cfg, st = capi.Weights(), capi.Config(), capi.RunState()
    hip.load_model(C.byref(w), C.byref(cfg), path.encode())
    most, V = 300, cfg.vocab_size
    cfg.max_seq_len = most
    hip.malloc_run_state(C.byref(st), C.byref(cfg))
    mgr = capi.KVCacheManager.in_dll(hip.dll, "g_kv_manager")
    hip.nvllm_set_kv_elem_bytes(4 if f32 or not folder else 2)
    hip.nvllm_init_model_kv(C.byref(mgr), 16, most, C.byref(cfg), C.byref(w))
    own = st.logits
    try:
        assert hip.nvllm_get_logits_mode() == 0
        tables, keep = (C.POINTER(capi.BlockTable) * most)(), []
        for i in range(most):
            at = (C.c_int * 1)(hip.alloc_block(C.byref(mgr)))
            keep.append((at, capi.BlockTable(C.cast(at, capi.c_int_p), 1)))
            tables[i] = C.pointer(keep[-1][1])

        def rows_of(n, address, ahead):
            rows = np.ctypeslib.as_array(C.cast(address, capi.c_float_p), shape=(n + 1, V))
            rows[:] = -7.0
            st.logits = address
            args = (capi.ints([(5 * i + 3) % V for i in range(n)]), n, capi.ints([0] * n), capi.ints(range(n)), capi.ints(range(n)), n)
            tail = (C.byref(cfg), C.byref(st), C.byref(w), tables)
            if ahead:
                out = (C.c_int * n)()
                assert hip.nvllm_forward_collect(hip.nvllm_forward_enqueue(*args, None, *tail), out, n) == n
            else:
                hip.transformer_batch(*args, *tail)
            assert (rows[n] == -7.0).all()       # nothing behind the last row
            return rows[:n].copy()

        for n in (1, 6, 7, 17, 64, 65, 113, 257):
            plain = np.empty((n + 1, V), np.float32)
            want = rows_of(n, own, True)
            assert np.isfinite(want).all() and (want != -7.0).any()
            np.testing.assert_array_equal(rows_of(n, own, False), want)
            np.testing.assert_array_equal(rows_of(n, own + 4, False), want)                  # no whole 16 bytes: copied
            np.testing.assert_array_equal(rows_of(n, plain.ctypes.data, False), want)        # a caller's own array: copied
    finally:
        st.logits = own
        hip.free_kv_cache_manager(C.byref(mgr))
        hip.free_run_state(C.byref(st))
        hip.nvllm_free_model(C.byref(w))
        hip.nvllm_set_compute_dtype(capi.COMPUTE_BF16)
