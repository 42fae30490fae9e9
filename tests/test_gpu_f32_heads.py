"""The attention kernels of fp32 rows at the sizes where their work splits: outputs of more columns than a workgroup has
threads, rows that are not whole float4s, keys around a block of 256; and linear attention whose state a workgroup holds in
its registers, at every number of dims per thread, portions around a batch of eight tokens."""
import ctypes as C

import numpy as np
import pytest

from nvllm_amd import capi
from tests import hybrid_oracle as O
from tests.test_gpu_hybrid_ops import filled, reference
from tests.test_gpu_latent_ops import Dev, filled_pool, reference_attention, rng, rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,vdim", [(20, 1100), (68, 516), (13, 300), (4, 4)])
def test_windowed_attention(hip, dim, vdim):
    lengths = [1, 255, 256, 257, 530]
    pool, kv = filled(hip, 1, dim, vdim, 4, 16, lengths, dim)
    seq, pos = list(range(5)), [n - 1 for n in lengths]
    q = rounded(rng(3).standard_normal((5, 2, dim)), 4)
    for size, keep, cap in ((1 << 30, 0, 5.0), (256, 1, 0.0)):
        got = pool.attend(seq, pos, q, 2.5 * dim ** -0.5, cap, size, keep)
        want = reference(kv, q, pos, seq, 2.5 * dim ** -0.5, cap, size, keep)
        assert np.abs(got - want).max() < 3e-5 * np.abs(want).max()   # the bar of the fp32 rows in test_gpu_hybrid_ops.py
    pool.close()


@pytest.mark.parametrize("rank,rot", [(1028, 8), (260, 4), (21, 6), (4, 4)])
def test_latent_attention(hip, rank, rot):
    lengths = [1, 255, 256, 257, 530]
    pool, rows_of = filled_pool(hip, rank, rot, 4, 16, lengths, rank)
    r = rng(5)
    seq, pos = list(range(5)), [n - 1 for n in lengths]
    q, sink, scale = rounded(r.standard_normal((5, 2, rank + rot)), 4), rounded(r.standard_normal(2), 4), 2.0 * (rank + rot) ** -0.5
    got = pool.attend(seq, pos, q, sink, scale)
    want = reference_attention(rows_of, q, pos, seq, sink, scale, rank)
    assert np.abs(got - want).max() < 3e-5 * np.abs(want).max()       # the bar of the fp32 rows in test_gpu_latent_ops.py
    pool.close()


@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 64), (64, 256), (256, 32), (128, 32), (128, 128)])
def test_linear_attention_of_portions(hip, dim, vdim):
    """4, 8 and 16 dims per thread, one to eight waves' lanes per row; a sequence's first tokens and later ones in one batch."""
    r = rng(dim + vdim)
    H, decay, cuts = 2, np.array([0.6, 0.99]), [[1, 7, 1], [8, 9, 16], [17, 1, 33]]
    data = [[rounded(r.standard_normal((sum(c), H, w)) * 0.7, 4) for w in (dim, dim, vdim)] for c in cuts]
    state = hip.to_device(np.asarray(r.standard_normal((3, H, dim, vdim)), np.float32))   # another sequence's remains
    got, at = [[] for _ in cuts], [0] * 3
    for step in range(3):
        ids, pos, parts = [], [], []
        for s, c in enumerate(cuts):
            ids += [s] * c[step]
            pos += list(range(at[s], at[s] + c[step]))
            parts.append([x[at[s]:at[s] + c[step]] for x in data[s]])
            at[s] += c[step]
        q, k, v = (np.concatenate(x) for x in zip(*parts))
        T, d = len(ids), Dev(hip)
        out = d.empty(T * H * vdim)
        hip.nvllm_lightning(out, None, d(q), d(k), d(v), None, None, (C.c_float * H)(*decay), state, capi.ints(ids), capi.ints(pos), H, dim, vdim, 4, T)
        o = hip.to_host(out, (T, H, vdim))
        d.close()
        for s in range(3):
            got[s].append(o[[i for i, x in enumerate(ids) if x == s]])
    have = hip.to_host(state, (3, H, dim, vdim))
    for s in range(3):
        o, st = O.decayed_state(*data[s], np.float32(decay).astype(np.float64))
        assert np.abs(have[s] - st).max() < 4e-6 * np.abs(st).max(), s       # the bars of test_gpu_hybrid_ops.py
        assert np.abs(np.concatenate(got[s]) - o).max() < 5e-6 * np.abs(o).max(), s
    hip.free(state)
