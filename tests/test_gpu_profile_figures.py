"""The bytes and operations that the kernel timing reports for the experts' products of fp32 rows: those of the pairs of a token
and a choice and of the experts they can reach, not of the padding the launch has room for; and for work that rides in another's launch:
beside that launch's own."""
import ctypes as C

import numpy as np
import pytest

from nvllm_amd import synth
from tests import hybrid_util, latent_util, util
from tests.test_gpu_latent_ops import Dev, rng

pytestmark = pytest.mark.gpu


def figures(hip):
    """(launches, bytes, operations) of every class since the last call."""
    got = {}
    for c in range(hip.nvllm_prof_num_classes()):
        n, ms, by, fl = C.c_longlong(), C.c_double(), C.c_double(), C.c_double()
        hip.nvllm_prof_get(c, C.byref(n), C.byref(ms), C.byref(by), C.byref(fl))
        if n.value:
            got[hip.nvllm_prof_name(c).decode()] = (n.value, by.value, fl.value)
    hip.nvllm_prof_reset()
    return got


def of_pass(hip, eng, util, plan, seqs):
    hip.nvllm_prof_reset()
    hip.nvllm_prof_enable(1)
    try:
        util.feed_all(eng, plan, seqs)
    finally:
        hip.nvllm_prof_enable(0)
    return figures(hip)


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
    got = figures(hip)
    d.close()
    pairs = T * top
    touched = min(E, pairs)
    assert got["gemm_expert_up"] == (1, 4.0 * (touched * 2 * ff * D + pairs * (D + ff)), 2.0 * pairs * 2 * ff * D)
    assert got["gemm_expert_down"] == (1, 4.0 * (touched * D * ff + pairs * (ff + D)), 2.0 * pairs * D * ff)


@pytest.mark.parametrize("T,f32", [(64, False), (300, False), (64, True)])   # streaming, tiles, fp32
def test_routing_beside_the_shared_expert(hip, tmp_path, T, f32):
    D, F, E, top = 288, 160, 16, 2
    cfg = synth.hybrid_config(D, 64, [(hybrid_util.A(4, 2, 16, 16, size=48, keep_first=4), hybrid_util.E(32, E, top, F))])
    path, _, _ = hybrid_util.model(tmp_path, "figures", cfg=cfg)
    eng = hybrid_util.engine(hip, path, f32, slots=1)
    got = of_pass(hip, eng, hybrid_util, [[(0, T)]], {0: hybrid_util.tokens(T, 64, 1)})
    eng.close()
    choice, sort = T * (4.0 * E + 20.0 * top), 28.0 * T * top
    assert "route" not in got and ("gemm_router" in got) == f32
    if f32:
        assert got["gemm_shared_up"] == (1, 4.0 * (2 * F * D + T * (D + F)) + choice, 2.0 * T * 2 * F * D)
        return
    chosen = T > 255   # beside the first product already
    router = 2.0 * (E + 1) * D + 4.0 * T * (E + 1)
    assert got["gemm_shared_up"] == (1, 2.0 * 2 * F * D + 2.0 * T * D + 1.0 * T * 2 * F + router + (choice if chosen else 0), 2.0 * T * D * (2 * F + E + 1))
    assert got["gemm_shared_down"] == (1, 2.0 * F * D + 2.0 * T * F + 4.0 * T * D + (sort if chosen else choice), 2.0 * T * F * D)


def test_forming_beside_single_tokens(hip, tmp_path):
    H, rank, dim = 24, 256, 64
    cfg = synth.latent_config(64, 130, [(synth.latent_mixer(H, dim, 64, dim, rank, 32), 40)] * 2, streams=2)
    path, _, _ = latent_util.model(tmp_path, "figures", cfg=cfg)
    seqs = {0: latent_util.tokens(32, 130, 1), 1: latent_util.tokens(600, 130, 2)}
    got = []
    for plan in ([[(0, 30)], [(0, 1), (1, 600)]], [[(0, 30)], [(0, 1)], [(1, 600)]]):   # beside each other, and apart
        eng = latent_util.engine(hip, path, False, slots=2)
        got.append(of_pass(hip, eng, latent_util, plan, seqs))
        eng.close()
    assert "latent_expand" not in got[0] and got[1]["latent_expand"][0] == 2
    for i in (1, 2):
        assert got[0]["latent_attn_tok"][i] == got[1]["latent_attn_tok"][i] + got[1]["latent_expand"][i]


@pytest.mark.parametrize("first,tokens", [(40, 1), (40, 30), (100, 700)])   # one row, a portion by 16 columns, one by 64
def test_paged_attention_operator(hip, first, tokens):
    heads, kv_heads, hd = 16, 4, 64
    hip.nvllm_set_kv_elem_bytes(2)
    try:
        pool = util.Pool(hip, 16, -(-(first + tokens) // 16), 1, kv_heads, hd)
        pool.new_table(-(-(first + tokens) // 16))
        pool.grow(0, first + tokens)
        rows = rng(1).standard_normal((first + tokens, kv_heads * hd)).astype(np.float32)
        util.op_kv_write_batch(hip, pool, rows, rows, 0, list(range(first + tokens)), [0] * (first + tokens), kv_heads, hd)
        hip.nvllm_prof_reset()
        hip.nvllm_prof_enable(1)
        util.op_paged_attention_batch(hip, pool, rng(2).standard_normal((tokens, heads * hd)).astype(np.float32), 0, list(range(first, first + tokens)), [0] * tokens,
                                      first + tokens, heads, kv_heads, hd)
    finally:
        hip.nvllm_prof_enable(0)
        hip.nvllm_set_kv_elem_bytes(4)
    got = figures(hip)
    pool.close()
    pairs = sum(range(first + 1, first + tokens + 1))
    assert got["attn"] == (1, (first + tokens) * 2.0 * kv_heads * hd * 2 + tokens * heads * hd * 8.0, 4.0 * pairs * heads * hd)
