"""Which passes' logits rows the classifier stores for the host itself: rows of a vocabulary that is no multiple of four, which cross value
by value, up to 32 of them; others in any number; none outside malloc_run_state's array or off its 16 bytes."""
import ctypes as C

import numpy as np
import pytest

from nvllm_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [32000, 32001, 32002, 32003, 203, 512])
def test_which_rows_are_stored(hip, vocab):
    cfg, st = capi.Config(), capi.RunState()
    cfg.dim, cfg.hidden_dim, cfg.n_layers, cfg.n_heads, cfg.n_kv_heads, cfg.vocab_size, cfg.max_seq_len, cfg.head_dim = 64, 64, 1, 1, 1, vocab, 65, 64
    hip.malloc_run_state(C.byref(st), C.byref(cfg))
    own = st.logits
    stored = hip.dll.nvllm_internal_rows_stored
    try:
        assert hip.nvllm_get_logits_mode() == 0
        for rows in (1, 31, 32, 33, 64):
            st.logits = own
            assert stored(C.byref(st), rows, vocab) == int(vocab % 4 == 0 or rows <= 32), rows
            st.logits = own + 4
            assert not stored(C.byref(st), rows, vocab)
            plain = np.empty(64 * vocab, np.float32)
            st.logits = plain.ctypes.data
            assert not stored(C.byref(st), rows, vocab)
        st.logits = own
        assert not stored(C.byref(st), 0, vocab) and not stored(C.byref(st), 66, vocab)   # (more rows than the array holds)
    finally:
        st.logits = own
        hip.free_run_state(C.byref(st))
