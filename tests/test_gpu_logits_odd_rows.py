"""Many logits rows of a vocabulary that is no multiple of four: no slower in malloc_run_state's array, where the classifier may store
them itself, than where a copy has to bring them."""
import ctypes as C
import time

import numpy as np
import pytest

from nvllm_amd import capi, synth

pytestmark = pytest.mark.gpu
ROWS, VOCAB = 64, 32003


def test_odd_rows_take_no_longer_than_a_copy(hip, tmp_path):
    path = str(tmp_path / "m.bin")
    synth.write_model(path, synth.ModelShape.named("stories42M", n_layers=1, vocab_size=VOCAB, max_seq_len=64), seed=3, dtype="f32", exact16=False)
    hip.nvllm_set_compute_dtype(capi.COMPUTE_F32)
    w, cfg, st = capi.Weights(), capi.Config(), capi.RunState()
    hip.load_model(C.byref(w), C.byref(cfg), path.encode())
    cfg.max_seq_len = ROWS + 1   # (the rows fit four bytes further on)
    hip.malloc_run_state(C.byref(st), C.byref(cfg))
    mgr = capi.KVCacheManager.in_dll(hip.dll, "g_kv_manager")
    hip.nvllm_set_kv_elem_bytes(4)
    hip.nvllm_init_model_kv(C.byref(mgr), 16, ROWS, C.byref(cfg), C.byref(w))
    own = st.logits
    try:
        assert hip.nvllm_get_logits_mode() == 0
        tables, keep = (C.POINTER(capi.BlockTable) * ROWS)(), []
        for i in range(ROWS):
            at = (C.c_int * 1)(hip.alloc_block(C.byref(mgr)))
            keep.append((at, capi.BlockTable(C.cast(at, capi.c_int_p), 1)))
            tables[i] = C.pointer(keep[-1][1])
        args = (capi.ints([(5 * i + 3) % VOCAB for i in range(ROWS)]), ROWS, capi.ints([0] * ROWS), capi.ints(range(ROWS)), capi.ints(range(ROWS)), ROWS,
                C.byref(cfg), C.byref(st), C.byref(w), tables)
        plain = np.empty((ROWS, VOCAB), np.float32)   # not page-locked: never stored to
        rows = np.ctypeslib.as_array(C.cast(own, capi.c_float_p), shape=(ROWS, VOCAB))
        hip.transformer_batch(*args)
        want = rows.copy()
        st.logits = plain.ctypes.data
        hip.transformer_batch(*args)
        np.testing.assert_array_equal(plain, want)
        seconds = {0: [], 4: []}
        for i in range(300):   # the page-locked array, and four bytes into it, from where rows are copied
            st.logits = own + 4 * (i & 1)
            at = time.perf_counter()
            hip.transformer_batch(*args)
            seconds[4 * (i & 1)].append(time.perf_counter() - at)
        stored, copied = np.median(seconds[0]), np.median(seconds[4])
        # both are copied now: within a percent; stored value by value a pass of 291 us took 8 % longer
        assert stored < 1.03 * copied, (stored, copied)
    finally:
        st.logits = own
        hip.free_kv_cache_manager(C.byref(mgr))
        hip.free_run_state(C.byref(st))
        hip.nvllm_free_model(C.byref(w))
        hip.nvllm_set_compute_dtype(capi.COMPUTE_BF16)
