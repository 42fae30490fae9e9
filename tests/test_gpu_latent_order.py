"""Single tokens before, between and behind prompt portions that form their keys and values (csrc/latent_prompt.hip): the same bits
wherever the scheduler puts them, and as few tokens through the products of the attention over latents."""
import ctypes as C

import numpy as np
import pytest

from nvllm_amd import capi, synth
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


def test_tokens_taken_from_the_pass_before(hip, tmp_path):
    """A pass sent ahead: rows between the prompts continue with the arg-max of the pass before, by the caller's own numbering."""
    hip.nvllm_set_compute_dtype(capi.COMPUTE_BF16)
    hip.nvllm_set_logits_mode(0)
    path, _, _ = U.model(tmp_path, "order", seed=5, cfg=CONFIG)
    w, cfg, st = capi.Weights(), capi.Config(), capi.RunState()
    hip.load_model(C.byref(w), C.byref(cfg), path.encode())
    cfg.max_seq_len = 2048
    hip.malloc_run_state(C.byref(st), C.byref(cfg))
    mgr = capi.KVCacheManager.in_dll(hip.dll, "g_kv_manager")
    hip.nvllm_set_kv_elem_bytes(2)
    hip.nvllm_init_model_kv(C.byref(mgr), 16, 2 * LONG // 16 + 3 * 8, C.byref(cfg), C.byref(w))
    try:
        tables, keep = (C.POINTER(capi.BlockTable) * 5)(), []
        for q in range(5):
            n = LONG // 16 if q in PROMPTS else 8
            at = (C.c_int * n)(*[hip.alloc_block(C.byref(mgr)) for _ in range(n)])
            keep.append((at, capi.BlockTable(C.cast(at, capi.c_int_p), n)))
            tables[q] = C.pointer(keep[-1][1])
        tail = (C.byref(cfg), C.byref(st), C.byref(w), tables)

        def rows_of(n):
            return np.ctypeslib.as_array(C.cast(st.logits, capi.c_float_p), shape=(n, cfg.vocab_size)).copy()

        lengths = {q: 70 + 9 * q for q in ROWS}
        got = []
        for ahead in (False, True):
            parts = [(q, U.tokens(lengths[q], 130, q)) for q in ROWS]
            ends = np.cumsum([len(t) for _, t in parts])
            args = [np.concatenate([t for _, t in parts]), np.concatenate([np.arange(len(t)) for _, t in parts]), np.concatenate([[q] * len(t) for q, t in parts]), ends - 1]
            hip.transformer_batch(capi.ints(args[0]), int(ends[-1]), capi.ints(args[1]), capi.ints(args[2]), capi.ints(args[3]), 3, *tail)
            best = rows_of(3).argmax(1)
            order = [3, 0, 2, 1, 4]
            tokens, pos, ids, src, out = [], [], [], [], []
            for q in order:
                if q in PROMPTS:
                    t = U.tokens(LONG, 130, q)
                    tokens += list(t)
                    pos += range(LONG)
                    ids += [q] * LONG
                    src += [-1] * LONG
                else:
                    tokens.append(0 if ahead else int(best[ROWS.index(q)]))
                    pos.append(lengths[q])
                    ids.append(q)
                    src.append(ROWS.index(q) if ahead else -1)
                out.append(len(tokens) - 1)
            out = out[::-1]   # output rows in an order of the caller's own
            args = (capi.ints(tokens), len(tokens), capi.ints(pos), capi.ints(ids), capi.ints(out), 5)
            if ahead:
                first = (C.c_int * 5)()
                assert hip.nvllm_forward_collect(hip.nvllm_forward_enqueue(*args, capi.ints(src), *tail), first, 5) == 5
                np.testing.assert_array_equal(np.array(first), rows_of(5).argmax(1))
            else:
                hip.transformer_batch(*args, *tail)
            got.append(rows_of(5))
        np.testing.assert_array_equal(got[1], got[0])
    finally:
        hip.free_kv_cache_manager(C.byref(mgr))
        hip.free_run_state(C.byref(st))
        hip.nvllm_free_model(C.byref(w))
