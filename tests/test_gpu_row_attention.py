"""Attention of single tokens over fp32 rows, one and two query heads on a key/value head: contexts that end inside a group of keys, at the
end of a trip and of two, and beyond; every head width."""
import pytest

from tests.test_gpu_slices import check_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,heads,kv_heads", [(16, 8, 8), (32, 8, 4), (48, 6, 6), (64, 8, 8), (64, 8, 4), (80, 4, 4), (96, 4, 2), (128, 4, 4), (128, 4, 2)])
@pytest.mark.parametrize("longest", [1, 2, 7, 16, 17, 63, 128, 129, 256, 257, 512, 513, 1030])
def test_rows(hip, hd, heads, kv_heads, longest):
    contexts = [longest, 1, max(1, longest - 3), max(1, longest // 2)]
    hip.nvllm_set_kv_elem_bytes(4)
    check_rows(hip, hd, heads, kv_heads, 4, longest, contexts)


@pytest.mark.parametrize("longest", [300, 1024, 1025])
def test_many_rows(hip, longest):   # items for every CU: up to 1,024 keys
    hip.nvllm_set_kv_elem_bytes(4)
    check_rows(hip, 64, 8, 8, 4, longest, [longest - 7 * (i % 5) for i in range(33)])
