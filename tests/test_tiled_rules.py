"""Which products of many rows are tiled ones, whole or as sums, and which merged
rows are converted at once: the rules of kubeai_amd/ops at shapes whose times on both
sides are known (us, weights out of cache)."""
import pytest
import torch

import kubeai_amd.ops as ops


@pytest.mark.parametrize("M,N,K,fp8,better", [
    # library / tiled
    (384, 28672, 4096, True, True),    # 60 / 45
    (2048, 28672, 4096, True, True),   # 228 / 211
    (97, 6144, 4096, True, False),     # 15.9 / 17.1
    (128, 6144, 4096, True, False),    # 16.1 / 18.1
    (148, 7168, 5632, True, True),     # 22.3 / 21.4
    (412, 3968, 9344, True, True),     # 43 / 33
    (775, 256, 11776, True, False),    # 15.9 / 32.7
    (570, 640, 6400, True, False),     # 16.1 / 23.5
    (119, 6144, 3072, True, False),    # 12.7 / 15.8
    (353, 1504, 18304, True, True),    # 77 / 56
    (256, 28672, 4096, True, False),   # 40.4 / 40.7
    (260, 28672, 4096, True, True),    # 56 / 43
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
    # few rows beside wide weights whose rows are no whole 4 KB
    (36, 96256, 2304, False, True),    # 95 / 86
    (67, 91392, 3264, False, True),    # 132 / 124
    (61, 57984, 1856, False, False),   # 42.9 / 45.5
    (29, 67072, 8000, False, False),
    (37, 98624, 640, False, True),     # 50 / 36
    (36, 22016, 1280, True, True),     # 11.7 / 10.2
    (40, 18432, 128, True, True),      # 5.2 / 4.8
    (40, 35840, 2048, True, False),    # 21.1 / 23.8
    (41, 33408, 1536, True, False),    # 18.1 / 19.7
    (72, 58816, 1024, True, True),     # 36.7 / 20.7
    (39, 54272, 256, True, False),     # 8.7 / 9.9
])
def test_whole_products(M, N, K, fp8, better):
    assert ops._tiled_better(M, N, K, fp8) is better


@pytest.mark.parametrize("M,N,K,better", [
    # library's product and activation / in one launch
    (128, 28672, 4096, True),    # 58.4 / 56.2
    (384, 28672, 4096, True),    # 88 / 83
    (640, 28672, 4096, False),   # 150 / 160
    (1024, 18432, 2304, True),   # 102 / 94
    (2048, 18432, 2304, False),  # 172 / 181
    (126, 9216, 7680, False),    # 53 / 60
    (121, 8448, 7168, False),    # 49 / 53
    (195, 17280, 6656, False),   # 82 / 91
    (208, 10624, 3840, False),   # 35 / 39
    (201, 11264, 2048, True),    # 31 / 22
    (96, 28672, 4096, False),
])
def test_activation_behind_the_product(M, N, K, better):
    assert ops.gated_better(M, N, K) is better


@pytest.mark.parametrize("n_q,splits,better", [
    # merge and conversion / in one launch, with the attention
    (16, 2, True),    # 13.2 / 10.9
    (16, 16, True),   # 16.0 / 14.3
    (32, 2, True),    # 13.9 / 13.1
    (32, 10, False),  # 14.2 / 15.9
    (32, 16, False),  # 13.9 / 17.8
    (64, 2, False),   # 12.1 / 14.0
    (64, 12, False),  # 13.7 / 24.7
    (8, 1, False),    # (nothing to merge)
])
def test_merged_rows_converted(n_q, splits, better):
    assert ops.decode_fp8_merges(n_q, splits) is better


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
    (128, 4096, 0, False, False),      # (nothing to add up: the library's zeros)
    (128, 0, 4096, True, False),
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
    (22, 896, 11008, True, False, False),   # streaming 12.6 / 13.3
    (23, 1920, 9344, False, False, False),  # streaming 16.6 / 17.1
    (18, 512, 17920, True, False, True),    # streaming 15.8 / 15.3
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


@pytest.mark.skipif(not ops.have_hip_ext(), reason="the costs are the extension's")
@pytest.mark.parametrize("rows,N,K,shapes", [
    # of 2048 x 1024 and 1024 x 1024, in tiles of 256 x 192: 81 us a layer, now 62
    (2646, 1024, 1024, (5, 6, 7)),
    (2646, 2048, 1024, (4, 5, 6)),
    (4176, 4096, 2560, (1,)),         # 81, now 60
    (4096, 28672, 4096, (0,)),
])
def test_tiles_of_eight_experts(rows, N, K, shapes):
    from kubeai_amd import _C

    shape, parts, _ = _C.tiled_plan(rows, N, K, True, False, experts=8)
    assert shape in shapes and parts == 1


@pytest.mark.parametrize("rows,N,K,fp8,better", [
    # each expert's rows: by themselves / all in one launch
    (512, 28672, 4096, True, True),
    (1024, 28672, 4096, False, True),    # 1664 / 1666
    (2048, 28672, 4096, False, False),   # 2907 / 3233
    (2048, 3584, 2048, False, True),     # 275 / 249
    (4096, 3584, 2048, False, False),    # 388 / 467
    (3772, 1280, 768, False, True),      # the layer 302 / 132
])
def test_experts_in_one_launch(rows, N, K, fp8, better):
    w = torch.empty(4, N, K, dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16, device="meta")
    assert ops.grouped_linear_better(4 * rows, w) is better


def test_no_rule_keeps_the_sizes_of_a_trace():
    class Reader(torch.nn.Module):
        def forward(self, x):
            assert ops.sums_for_reader(x, torch.zeros(64, 14336)) is None
            return x + 1

    before = ops.tiled_sums_better.cache_info().currsize
    torch.jit.trace(Reader(), torch.randn(128, 14336), check_trace=False)
    assert ops.tiled_sums_better.cache_info().currsize == before


@pytest.mark.gpu
@pytest.mark.parametrize("rows,taken", [(8, True), (40, True), (64, True), (128, False)])
def test_no_rule_keeps_them_with_operands_that_tiles_take(rows, taken):
    class Reader(torch.nn.Module):
        def forward(self, x):
            ops.sums_for_reader(x, w)
            return x + 1

    w = torch.randn(2304, 9216, device="cuda").bfloat16()
    x = torch.randn(rows, 9216, device="cuda").bfloat16()
    rules = (ops.narrow_better, ops.tiled_sums_better)
    ops.sums_for_reader(x, w)
    before = [rule.cache_info().currsize for rule in rules]
    for _ in range(2):
        torch.jit.trace(Reader(), x, check_trace=False)
    assert [rule.cache_info().currsize for rule in rules] == before
    assert ops.narrow_better(rows, 2304, 9216, False) is taken
