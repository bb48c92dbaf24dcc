"""Which product goes where: the rules of kubeai_amd/ops at shapes whose times
on both sides are known (weights out of cache, replayed from a graph)."""
import pytest

from kubeai_amd.ops import _streams_better, sums_better


@pytest.mark.parametrize("M,N,K,fp8,better", [
    # wide weights: library / streaming, us
    (8, 28672, 4096, False, True),    # 60.2 / 41.0
    (16, 18432, 2304, False, True),   # 50.4 / 22.3
    (8, 32256, 2048, False, True),    # 32.5 / 25.0
    (1, 16384, 512, False, True),     # 11.5 / 5.8
    (8, 16384, 4096, False, True),    # 32.1 / 23.5
    (1, 16384, 8192, False, True),    # 61.2 / 46.9
    (8, 24576, 8192, False, True),    # 81.9 / 70.6
    (16, 22528, 6144, False, True),   # 64.2 / 60.3
    (8, 20480, 6144, False, True),    # 103 / 53
    (8, 36864, 8192, False, True),    # 132 / 116
    (8, 65536, 4096, False, True),    # 125 / 91
    (8, 16384, 4096, True, True),     # 26.4 / 14.0
    (16, 30720, 8192, True, True),    # 61.5 / 44.4
    (8, 36864, 4096, True, True),     # 38.2 / 32.5
    (8, 65536, 128, True, False),     # 5.4 / 5.1
    (17, 28672, 4096, True, False),   # (the tiled product's)
    (8, 128256, 4096, False, True),   # 187 / 173
    (8, 256000, 2304, False, False),  # 207 / 218
    # even shares of the columns, and beside them
    (8, 49152, 1280, False, True),    # 31.7 / 26.3
    (8, 49152, 2304, False, True),    # 48.9 / 43.7
    (13, 49536, 2304, False, False),  # 43.3 / 50.8
    (10, 49152, 4320, False, False),
    (8, 49152, 5120, True, True),     # 49.2 / 48.5
    (13, 53504, 1920, True, False),   # 21.7 / 23.1
    (8, 81920, 2304, True, False),
    (12, 51008, 704, True, True),     # 19.4 / 10.9
    # cut along K
    (8, 9216, 6656, True, True),      # 38 / 19
    (16, 8192, 8192, True, False),    # 16.4 / 21.3
    (8, 14848, 7680, False, False),   # 45 / 52
    # long rows
    (32, 2048, 32256, False, True),   # 111 / 32
    (96, 4096, 40960, True, True),    # 139 / 55
    (16, 1024, 16384, False, True),   # 21.0 / 16.4
    (48, 1024, 16384, False, False),  # 21.3 / 19.2
    (33, 512, 16384, False, False),   # 18.7 / 16.8
    (64, 1024, 16384, True, True),    # 26.4 / 14.5
    (96, 2048, 16384, True, False),   # 21.6 / 17.5
    (8, 4096, 14336, False, False),   # 25.8 / 27.2
])
def test_streaming_products(M, N, K, fp8, better):
    assert _streams_better(M, N, K, fp8) is better


@pytest.mark.parametrize("M,N,K,fp8,rope,better", [
    # with the norm that reads the product: library / sums, us
    (8, 4096, 4096, False, False, True),     # 18.9 / 13.5
    (96, 4096, 4096, False, False, True),    # 25.3 / 19.3
    (40, 4096, 14336, False, False, True),   # 39.4 / 32.1
    (8, 1024, 8192, False, False, True),     # 14.6 / 12.3
    (40, 1024, 8192, False, False, False),   # 15.3 / 12.4: the tiled product's sums
    (8, 8192, 8192, False, False, False),    # 34.7 / 41.4
    (17, 12288, 8192, False, False, False),  # 45.8 / 55.1
    (96, 5120, 2048, False, False, False),   # 17.2 / 19.6
    (8, 10240, 1024, False, False, True),    # 0.93 of the library's
    (8, 4608, 28672, False, False, True),    # 0.47
    (16, 4096, 4096, True, False, True),     # 15.8 / 13.3
    (64, 4096, 4096, True, False, False),    # 16.6 / 15.4: a cautious line
    (40, 4096, 14336, True, False, True),    # 25.1 / 22.8
    (8, 8192, 8192, True, False, True),      # 47.5 / 26.6
    (16, 8192, 8192, True, False, False),    # 20.6 / 27.2
    (40, 8192, 8192, True, False, False),    # 22.9 / 28.5
    (8, 4096, 512, True, False, False),      # 8.6 / 7.2: the same
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
