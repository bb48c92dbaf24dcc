"""Which product goes where: the rules of kubeai_amd/ops at shapes whose times
on both sides are known (weights out of cache, replayed from a graph)."""
import pytest

from kubeai_amd.ops import _streams_better


@pytest.mark.parametrize("M,N,K,fp8,better", [
    # wide weights: library / streaming, us
    (8, 28672, 4096, False, True),    # 59.9 / 47.6
    (16, 18432, 2304, False, True),   # 50.6 / 25.7
    (8, 32256, 2048, False, True),    # 34.5 / 31.4
    (1, 16384, 512, False, True),     # 11.5 / 6.5
    (8, 16384, 4096, False, False),   # 33.4 / 34.8
    (1, 16384, 8192, False, False),   # 64.7 / 67.7
    (8, 24576, 8192, False, False),   # 83.8 / 91.8
    (16, 22528, 6144, False, False),  # 67.4 / 75.5
    (8, 20480, 6144, False, True),    # 104 / 64
    (8, 36864, 8192, False, False),   # 145 / 160
    (8, 65536, 4096, False, True),    # 123 / 107
    (8, 16384, 4096, True, True),     # 27.9 / 20.3
    (16, 30720, 8192, True, True),    # 66 / 57
    (8, 36864, 4096, True, False),    # 41.4 / 42.7
    (8, 65536, 128, True, False),     # 5.6 / 6.7
    (17, 28672, 4096, True, False),   # 29.4 / 30.7
    (8, 128256, 4096, False, False),  # 192 / 198
    # long rows
    (32, 2048, 32256, False, True),   # 111 / 38
    (96, 4096, 40960, True, True),    # 140 / 58
    (16, 1024, 16384, False, True),   # 21.1 / 19.4
    (48, 1024, 16384, False, False),  # 21.0 / 28.7
    (33, 512, 16384, False, False),   # 19.0 / 27.7
    (64, 1024, 16384, True, True),    # 26.2 / 19.9
    (96, 2048, 16384, True, False),   # 21.2 / 22.2
    (8, 4096, 14336, False, False),   # 27 / 29
])
def test_streaming_products(M, N, K, fp8, better):
    assert _streams_better(M, N, K, fp8) is better
