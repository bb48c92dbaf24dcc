"""Decode attention at the edges of its tiles (16-key blocks, tiles of 32 keys
at head size 128, 4 waves, splits) and of its group sizes.

The weights keep fp32 accuracy, so the bound is the output's own rounding to
bf16 (2^-9 of itself) plus fp32 sums and exponentials (1e-5 of max|v| ~ 5);
twice that is allowed."""
import pytest
import torch

import kubeai_amd.ops as ops
from kubeai_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(lens, nq, nkv, hd, scale, window=0, softcap=0.0, fp8=False, spare=0):
    torch.manual_seed(sum(lens) + nq * hd)
    need = [(n + 15) // 16 for n in lens]
    nb = sum(need) + 1
    order = torch.randperm(nb - 1) + 1
    bt = torch.zeros(len(lens), max(need) + spare, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = order[at : at + n]
        at += n
    kc = torch.randn(nb, nkv, 16, hd, device=DEV, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    for i, n in enumerate(lens):  # rows behind the last key hold anything
        if n % 16:
            kc[bt[i, need[i] - 1], :, n % 16 :] = float("nan")
            vc[bt[i, need[i] - 1], :, n % 16 :] = float("nan")
    if fp8:
        kc, vc = kc.to(torch.float8_e5m2), vc.to(torch.float8_e5m2)
    q = torch.randn(len(lens), nq + 2, hd, device=DEV, dtype=torch.bfloat16)[:, :nq]
    total = torch.tensor(lens, dtype=torch.int32, device=DEV)
    got = ops.paged_attention_decode(q, kc, vc, bt.to(DEV), total, scale, window=window,
                                     softcap=softcap)
    want = ref.paged_attention_decode(q.float(), kc.float(), vc.float(), bt.to(DEV), total,
                                      scale, window=window, softcap=softcap)
    torch.testing.assert_close(got.float(), want, atol=1e-4, rtol=2.0 ** -8)


EDGES = [1, 15, 16, 17, 31, 32, 33, 64, 127, 128, 129, 161, 700, 2049]


@pytest.mark.parametrize("group", [1, 2, 4, 5, 6, 8])
@pytest.mark.parametrize("hd", [128, 256])
def test_lengths_and_groups(group, hd):
    _run(EDGES, 2 * group, 2, hd, hd ** -0.5)


@pytest.mark.parametrize("rows", [1, 3, 600])
def test_one_split_and_many(rows):
    # 600 rows of one kv head are not split, one row is split sixteen times
    _run([5 + 37 * i % 300 for i in range(rows)], 4, 1, 128, 0.09, spare=50)


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("window", [1, 16, 31, 33, 500])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_windows(hd, window, softcap):
    _run(EDGES, 4, 2, hd, hd ** -0.5, window=window, softcap=softcap)


@pytest.mark.parametrize("hd", [128, 256])
def test_eight_bit_cache(hd):
    _run(EDGES, 8, 2, hd, hd ** -0.5, fp8=True)


def test_peaked_flat_and_negative_scales():
    _run(EDGES, 8, 2, 128, 3.0)
    _run(EDGES, 8, 2, 128, 0.0)
    _run(EDGES, 8, 2, 128, -0.2)


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_keys_that_are_not_finite(hd, softcap):
    """A NaN score reaches the output; a capped infinite one is the cap."""
    torch.manual_seed(hd)
    kc = torch.randn(9, 1, 16, hd, device=DEV, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    kc[2, 0, 5, 7] = float("nan")
    kc[4, 0, 3, 1], kc[6, 0, 3, 1] = float("inf"), -float("inf")
    bt = torch.tensor([[1, 2], [3, 4], [5, 6], [7, 8]], dtype=torch.int32, device=DEV)
    total = torch.full((4,), 30, dtype=torch.int32, device=DEV)
    q = torch.randn(4, 2, hd, device=DEV, dtype=torch.bfloat16)
    args = (bt, total, hd ** -0.5)
    got = ops.paged_attention_decode(q, kc, vc, *args, softcap=softcap).float()
    want = ref.paged_attention_decode(q.float(), kc.float(), vc.float(), *args, softcap=softcap)
    assert want[0].isnan().all() and want[3].isfinite().all()
    if softcap:
        torch.testing.assert_close(got, want, atol=1e-4, rtol=2.0 ** -8, equal_nan=True)
    else:  # an infinite score outweighs all others or is outweighed
        assert torch.equal(got.isnan(), want.isnan())


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e5m2])
@pytest.mark.parametrize("L", [1, 20, 300])
def test_values_that_are_not_finite(hd, cache, L):
    """An infinite value is infinite in the output, also behind a weight that bf16
    holds exactly (1 key: weight 1; equal scores: a power of two)."""
    torch.manual_seed(L)
    nb = (L + 15) // 16
    kc = torch.randn(3 * nb, 2, 16, hd, device=DEV, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    at = min(L - 1, 9)
    vc[0, 0, at, 3], vc[0, 0, at, 9], vc[0, 1, at, hd - 1] = float("inf"), -float("inf"), float("nan")
    vc[nb, 1, 0, 0] = float("inf")
    kc, vc = kc.to(cache), vc.to(cache)
    if cache != torch.bfloat16:  # (the conversion keeps infinities)
        assert vc[0, 0, at, 3].float().isinf()
    bt = torch.arange(3 * nb, dtype=torch.int32, device=DEV).view(3, nb)
    total = torch.full((3,), L, dtype=torch.int32, device=DEV)
    for scale in (hd ** -0.5, 0.0):
        q = torch.randn(3, 4, hd, device=DEV, dtype=torch.bfloat16)
        got = ops.paged_attention_decode(q, kc, vc, bt, total, scale).float()
        want = ref.paged_attention_decode(q.float(), kc.float(), vc.float(), bt, total, scale)
        assert want[0, 0, 3] == float("inf") and want[0, 1, 9] == -float("inf")
        torch.testing.assert_close(got, want, atol=1e-4, rtol=2.0 ** -8, equal_nan=True)


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("rows,n_kv,blocks", [(1, 1, 1), (1, 8, 4), (3, 4, 600), (32, 4, 250),
                                              (64, 4, 400), (128, 4, 500), (700, 2, 40)])
def test_splits(hd, rows, n_kv, blocks):
    """Two workgroups a CU where the rows allow it, never more splits than 16 or
    than a row can have tiles; many rows of head size 256 are split even where
    they fill the chip (a longer one among them would be worked through alone)."""
    from kubeai_amd import _C

    n = _C.paged_decode_splits(rows, n_kv, hd, blocks)
    tiles = blocks if hd == 256 else (blocks + 1) // 2
    assert 1 <= n <= min(16, tiles)
    assert n == min(16, tiles) or rows * n_kv * n >= 512
    assert n == 1 or rows * n_kv * (n - 1) < 576
    if hd == 256 and rows * n_kv == 512:
        assert n == 2


@pytest.mark.parametrize("group", [1, 2, 8])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e5m2])
def test_one_long_row_among_short_ones(group, cache):
    _run([3000] + [9] * 70, 2 * group, 2, 256, 0.06, fp8=cache != torch.bfloat16)


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("spread", [0.2, 0.7, 2.5])
def test_softcap_on_both_sides_of_its_forms(hd, spread):
    """Scores about and on both sides of 0.7 of the cap, where the form changes."""
    _run([70, 33], 4, 2, hd, spread * 20.0 * hd ** -0.5, softcap=20.0)


@pytest.mark.parametrize("rows,n_q,n_kv,hd", [
    (1, 8, 8, 128), (1, 4, 2, 128), (6, 20, 4, 128), (34, 32, 8, 256), (3, 32, 8, 128), (40, 32, 8, 128), (9, 40, 8, 128), (5, 128, 16, 128),
    (2, 136, 17, 128), (7, 8, 4, 256), (4, 16, 16, 256), (96, 32, 8, 128),
])
def test_fp8_rows_are_the_converted_bf16_rows(rows, n_q, n_kv, hd):
    """Merged and converted in one launch (up to 32 heads, few splits) or in two:
    the same bytes and scales."""
    torch.manual_seed(rows + n_q)
    lens = [int(x) for x in torch.randint(1, 900, (rows,))]
    lens[0] = 900
    width = (max(lens) + 15) // 16
    nb = rows * width + 1
    kc, vc = (torch.randn(nb, n_kv, 16, hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    bt = (torch.randperm(nb - 1)[: rows * width] + 1).int().view(rows, width).to(DEV)
    total = torch.tensor(lens, device=DEV, dtype=torch.int32)
    q = torch.randn(rows, n_q, hd, device=DEV, dtype=torch.bfloat16)
    got, scale = ops.paged_attention_decode_fp8(q, kc, vc, bt, total, hd ** -0.5)
    out = ops.paged_attention_decode(q, kc, vc, bt, total, hd ** -0.5)
    want, want_scale = ops.quant_fp8(out.view(rows, -1))
    assert torch.equal(scale, want_scale)
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))


def test_rows_of_a_larger_buffer():
    torch.manual_seed(0)
    kc, vc = (torch.randn(9, 2, 16, 128, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    bt = torch.arange(1, 9, dtype=torch.int32, device=DEV).view(2, 4)
    total = torch.tensor([60, 33], device=DEV, dtype=torch.int32)
    q = torch.randn(2, 8, 128, device=DEV, dtype=torch.bfloat16)
    out = torch.full((5, 8, 128), 7.0, device=DEV, dtype=torch.bfloat16)
    assert ops.paged_attention_decode(q, kc, vc, bt, total, 0.1, out=out) is out
    assert torch.equal(out[:2], ops.paged_attention_decode(q, kc, vc, bt, total, 0.1))
    assert (out[2:] == 7).all()


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("fp8", [False, True])
def test_last_tiles_of_a_wave(hd, fp8):
    """1 to 12 tiles a wave, even and odd, beside waves of none; what lies in the blocks
    behind a row's last one is not read. (A wave's tiles are every fourth of a split.)"""
    torch.manual_seed(hd)
    lens = [1, 16, 17, 32, 33, 63, 65, 127, 129, 191, 255, 257, 300, 400, 500, 700, 1100, 1501]
    nq, nkv, wide = 8, 2, 100
    need = [(n + 15) // 16 for n in lens]
    kc = torch.randn(sum(need) + 1, nkv, 16, hd, device=DEV, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    kc[0], vc[0] = float("nan"), float("nan")  # the table's other entries
    if fp8:
        kc, vc = kc.to(torch.float8_e5m2), vc.to(torch.float8_e5m2)
    bt = torch.zeros(len(lens), wide, dtype=torch.int32)
    at = 1
    for i, n in enumerate(need):
        bt[i, :n] = torch.arange(at, at + n)
        at += n
    for rows in ([len(lens) - 1], range(len(lens)), list(range(len(lens))) * 8):
        rows = list(rows)
        q = torch.randn(len(rows), nq, hd, device=DEV, dtype=torch.bfloat16)
        sl = torch.tensor([lens[i] for i in rows], dtype=torch.int32, device=DEV)
        args = (bt[rows].to(DEV), sl, hd ** -0.5)
        got = ops.paged_attention_decode(q, kc, vc, *args)
        want = ref.paged_attention_decode(q.float(), kc.float(), vc.float(), *args)
        # fp32 throughout, one rounding
        torch.testing.assert_close(got.float(), want, rtol=2.0 ** -8, atol=2.0 ** -9)
