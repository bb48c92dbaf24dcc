"""Which product goes where: the rules of kubeai_amd/ops at shapes whose times
on both sides are known (weights out of cache, replayed from a graph)."""
import pytest

from kubeai_amd.ops import _streams_better, sums_better


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


@pytest.mark.parametrize("M,N,K,fp8,rope,better", [
    # with the norm that reads the product: library / sums, us
    (8, 4096, 4096, False, False, True),     # 18.9 / 13.5
    (96, 4096, 4096, False, False, True),    # 25.3 / 19.3
    (40, 4096, 14336, False, False, True),   # 39.4 / 32.1
    (8, 1024, 8192, False, False, True),     # 14.6 / 12.3
    (40, 1024, 8192, False, False, False),   # 15.1 / 17.1
    (8, 8192, 8192, False, False, False),    # 34.7 / 41.4
    (17, 12288, 8192, False, False, False),  # 45.8 / 55.1
    (96, 5120, 2048, False, False, False),   # 17.2 / 19.6
    (8, 10240, 1024, False, False, True),    # 0.93 of the library's
    (8, 4608, 28672, False, False, True),    # 0.47
    (16, 4096, 4096, True, False, True),     # 15.8 / 13.3
    (64, 4096, 4096, True, False, False),    # 16.4 / 18.3
    (40, 4096, 14336, True, False, True),    # 25.1 / 22.8
    (8, 8192, 8192, True, False, True),      # 47.5 / 26.6
    (16, 8192, 8192, True, False, False),    # 20.6 / 27.2
    (40, 8192, 8192, True, False, False),    # 22.9 / 28.5
    (8, 4096, 512, True, False, False),      # 8.2 / 8.8
    (96, 2048, 2048, True, False, False),    # 11.7 / 11.5
    (40, 2304, 9216, True, False, True),     # 0.98
    # with the rotation and cache write
    (8, 6144, 4096, False, True, True),      # 0.88
    (64, 6144, 4096, False, True, False),    # 1.04
    (12, 6144, 4096, True, True, True),      # 0.52
    (64, 6144, 4096, True, True, False),     # 1.17
    (40, 6144, 4096, True, True, True),      # 1.03; a whole step 1104 with the library, 1089
    (40, 7168, 4096, True, True, False),     # 1.25
    (8, 1536, 512, True, True, False),       # 1.20
])
def test_products_as_sums(M, N, K, fp8, rope, better):
    assert sums_better(M, N, K, fp8, rope) is better
