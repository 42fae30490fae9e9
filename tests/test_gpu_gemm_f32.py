"""Projections of fp32 weights (matmul on a plain buffer) against 64-bit sums, at the sizes where the tiles end."""
import numpy as np
import pytest

from nvllm_amd import synth
from tests import hybrid_oracle as O
from tests import hybrid_util as U
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,N", [
    (1, 4, 1), (1, 288, 288), (16, 32, 16), (17, 36, 15),     # one token block and the first of the second; K past its last whole step
    (32, 100, 4100), (33, 512, 1376), (48, 64, 40),            # one and two row blocks, two token blocks
    (301, 512, 4128), (65, 1028, 8200),                        # four token blocks, ragged
    (1, 7, 5), (9, 130, 37), (5, 1, 3),                        # rows that are no multiples of 16 bytes
])
def test_matmul_on_fp32_weights(hip, T, K, N):
    rng = np.random.default_rng(T * 7 + K * 3 + N)
    x, w = rng.standard_normal((T, K)).astype(np.float32), rng.standard_normal((N, K)).astype(np.float32)
    got = util.op_matmul(hip, x, w)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    # a sum of K products in any order: K roundings of at most half a unit each, of the sum of magnitudes
    bound = (K + 2) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    assert (np.abs(got - x64 @ w64.T) <= bound).all()


def test_rows_beyond_the_sixteen_byte_grid_of_a_caller(hip):
    """A caller's pointer into the middle of a buffer."""
    rng = np.random.default_rng(3)
    T, K, N = 3, 64, 20
    x, w = rng.standard_normal((T, K)).astype(np.float32), rng.standard_normal((N, K)).astype(np.float32)
    dx, dw, do = hip.to_device(np.concatenate([np.zeros(1, np.float32), x.reshape(-1)])), hip.to_device(w), hip.empty_device(T * N * 4 + 4)
    hip.matmul(do + 4, dx + 4, dw, T, K, N)
    got = hip.to_host(do + 4, (T, N))
    for p in (dx, dw, do):
        hip.free(p)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    assert (np.abs(got - x64 @ w64.T) <= (K + 2) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)).all()


@pytest.mark.parametrize("T,K,N", [(3, 288, 768), (2, 512, 16500), (20, 512, 512), (40, 288, 3000), (300, 512, 768), (300, 288, 3000), (16, 1376, 512)])
def test_no_further_from_64_bits_than_64_chains(hip, T, K, N):
    """One block and several, K in eight and in four slices: the error of sums in 64 chains that meet in a tree, or near it."""
    rng = np.random.default_rng(T + K)
    x, w = rng.standard_normal((T, K)).astype(np.float32), (rng.standard_normal((N, K)) * K ** -0.5).astype(np.float32)
    got = util.op_matmul(hip, x, w)
    at = rng.integers(0, T, 16384), rng.integers(0, N, 16384)
    a, b = x[at[0]].astype(np.float64), w[at[1]].astype(np.float64)
    want = (a * b).sum(1)
    chains = np.zeros((16384, 64), np.float32)
    for k in range(0, K, 64):   # (a product of two fp32 numbers is exact in 64 bits)
        n = min(64, K - k)
        chains[:, :n] = a[:, k:k + n] * b[:, k:k + n] + chains[:, :n]
    while chains.shape[1] > 1:
        half = chains.shape[1] // 2
        chains = chains[:, :half] + chains[:, half:]
    # roundings counted: chains of eight with sums over each step come to 1.06 of it at K = 288, less above; chains of 16 to 1.17 at 512
    assert np.linalg.norm(got[at] - want) < 1.1 * np.linalg.norm(chains[:, 0] - want)


# three token blocks by two row blocks, in one round by eight waves and in several by four, and four token blocks by eight waves; ends of tiles
# and a K that is no multiple of a step or of the waves' share
@pytest.mark.parametrize("T,K,N", [(80, 1024, 2816), (289, 516, 500), (170, 1028, 2816), (200, 512, 1536), (193, 260, 1530), (230, 1024, 5632), (301, 512, 1536)])
def test_three_and_four_token_blocks(hip, T, K, N):
    test_matmul_on_fp32_weights(hip, T, K, N)
    test_no_further_from_64_bits_than_64_chains(hip, T, K, N)


@pytest.mark.parametrize("width,hidden,n", [(288, 768, 200), (512, 1376, 161)])
def test_pairs_of_three_token_blocks(hip, tmp_path, width, hidden, n):
    window = synth.window_mixer(4, 2, 16, 16, size=48, keep_first=4)
    cfg = synth.hybrid_config(width, 211, [(window, synth.expert_mlp(48, 4, 2, hidden))])
    path, cfg, weights = U.model(tmp_path, "pairs", seed=n, cfg=cfg)
    eng = U.engine(hip, path, True, slots=1)
    seq = U.tokens(n, 211, n)
    assert U.error(U.feed_all(eng, [[(0, n)]], {0: seq})[0], O.forward(cfg, weights, seq)) < U.limit(True)
    eng.close()
