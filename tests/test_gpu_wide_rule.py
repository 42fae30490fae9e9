"""Which launches take the 256-feature tiles of bf16 models (csrc/gemm_wide_b16.hip), and at which height: the sizes whose times stand
beside the rules, and their neighbours.  (256 CUs.)"""
import os

import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.skipif("NVLLM_GEMM_WIDE" in os.environ, reason="the environment forces a height")]


@pytest.mark.parametrize("N,K,T,height", [
    (4864, 2048, 700, 0), (3328, 2048, 1024, 0), (6656, 2048, 512, 0),       # four blocks on 209, 208, 208 CUs
    (5632, 2048, 700, 4), (6656, 2048, 528, 4),                              # ... on 242 and 234
    (6656, 2048, 640, 5), (4864, 2048, 1024, 5), (13312, 2048, 380, 6),      # 208, 247, 208
    (6656, 2048, 1024, 8), (6656, 2048, 1280, 10), (6656, 2048, 1536, 12), (6656, 2048, 1792, 14), (13312, 2048, 1024, 16),   # 208
    (11264, 2048, 1029, 14), (6656, 992, 1024, 0), (13312, 2048, 1152, 0)])  # a pass of prompts; a short K; more than a round at any height
def test_heights(hip, N, K, T, height):
    assert hip.dll.nvllm_internal_wide_height(N, K, T) == height
