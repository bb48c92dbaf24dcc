"""Which products of many rows are tiled ones, whole or as sums: the rules of
kubeai_amd/ops at shapes whose times on both sides are known (us, weights out
of cache)."""
import pytest

import kubeai_amd.ops as ops


@pytest.mark.parametrize("M,N,K,fp8,better", [
    # library / tiled
    (384, 28672, 4096, True, True),    # 60 / 45
    (2048, 28672, 4096, True, True),   # 228 / 211
    (97, 6144, 4096, True, True),
    (96, 6144, 4096, True, False),     # 14.0 / 16.1
    (640, 4096, 14336, True, True),    # 72 / 70
    (256, 4096, 14336, True, False),   # 34 / 49
    (160, 2304, 9216, True, False),    # 16 / 22
    (8192, 16384, 512, True, False),   # 104 / 127
    (160, 1024, 1024, True, False),    # 4.8 / 5.8
    (40, 128256, 4096, True, True),    # 129 / 107
    (16, 128256, 4096, True, False),
    (40, 57344, 8192, True, True),     # 121 / 103
    (40, 57344, 8192, False, False),
    (96, 128256, 4096, False, True),   # 225 / 207
    (2048, 28672, 4096, False, False),  # 333 / 391
    (2048, 128256, 4096, False, False),
])
def test_whole_products(M, N, K, fp8, better):
    assert ops._tiled_better(M, N, K, fp8) is better


@pytest.mark.skipif(not ops.have_hip_ext(), reason="the costs are the extension's")
@pytest.mark.parametrize("M,N,K,fp8,better", [
    # with the norm that reads the product: whole / sums
    (128, 4096, 14336, True, True),    # 51 / 26
    (384, 4096, 14336, True, True),    # 56 / 41
    (128, 4096, 4096, True, False),    # 15.5 / 16.7
    (128, 4096, 4096, False, True),    # library 28 / 19
    (2048, 4096, 14336, True, False),  # 114 / 127
    (1024, 4096, 4096, True, False),   # 26 / 36
    (160, 4096, 14336, False, True),   # library 86 / 38
    (1024, 4096, 14336, False, True),  # library 138 / 117
    (1024, 4096, 4096, False, False),  # library 47 / 50
    (512, 28672, 4096, True, False),   # (too wide for a norm)
    (160, 4096, 4000, False, False),   # (no whole steps of K)
    (96, 4096, 14336, True, False),    # (the streaming product's)
    (2049, 4096, 14336, False, False),
])
def test_products_as_sums(M, N, K, fp8, better):
    assert ops.tiled_sums_better(M, N, K, fp8) is better


@pytest.mark.parametrize("M,N,K,fp8,rope,better", [
    # with the reader: the best other form / tiled sums
    (24, 4096, 14336, True, False, True),   # 23.3 / 20.7
    (24, 4096, 4096, True, False, False),   # 13.0 / 14.2
    (40, 4096, 4096, True, False, True),    # streaming 15.4 / 13.4
    (40, 6144, 4096, True, True, True),     # 16.4 / 15.2
    (24, 2048, 2048, True, False, False),   # 8.8 / 9.8
    (96, 2048, 2048, True, False, False),   # library 12.3 / 11.2
    (40, 8192, 8192, True, False, False),   # 22.6 / 24.7
    (96, 4096, 4096, False, False, True),   # 19.8 / 17.2
    (96, 6144, 4096, False, True, True),    # 25.4 / 20.8
    (40, 8192, 28672, False, False, True),  # 108 / 88
    (80, 2304, 2048, False, False, False),  # 12.0 / 12.6
])
def test_few_rows_as_tiled_sums(M, N, K, fp8, rope, better):
    sums = ops.sums_better(M, N, K, fp8, rope)
    assert ops.few_tiled_better(M, N, K, fp8, rope, sums) is better
