"""Which kernel takes a projection, by its sizes: points on both sides of each rule, with the times beside the rules."""
import pytest

from k8s_llm_monitor_amd.ops import hybrid as hops


@pytest.mark.parametrize("M,N,K,f,takes", [
    (7830, 13312, 2048, 5632, True), (3749, 13312, 2048, 5632, True), (256, 53248, 2048, 26624, True), (1300, 53248, 2048, 0, True),
    (1, 53248, 2048, 26624, False), (64, 102400, 1024, 0, False), (128, 57344, 8192, 28672, False),  # a decode step's rows
    (300, 53248, 2048, 26624, False),  # two row tiles, little more than half full
    (50000, 288, 1024, 144, False),  # the same of features
    (6403, 4096, 1024, 0, True), (1300, 13312, 2048, 0, False),  # a last round that is half full, mostly empty
])
def test_tile_gemm_with_a_unit(M, N, K, f, takes):
    assert hops._tile_form(M, N, K, f) is takes
