"""Projections of fp32 weights (matmul on a plain buffer) against 64-bit sums, at the sizes where the tiles end."""
import numpy as np
import pytest

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
