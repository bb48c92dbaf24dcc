"""Prompt attention at the edges of its tiles: 32 rows a wave, 32 to 128 rows
a workgroup, 32 or 64 keys a staged tile, 16 tokens a cache block.

Bound: weights are rounded to bf16 before the second product (2^-9 of the
weighted sum of |v|, so 2^-9 max|v|), the output once more (2^-9 of itself);
the rest is fp32. Twice that is allowed."""
import pytest
import torch

import kubeai_amd.ops as ops
from kubeai_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(lens, ctxs, nq, nkv, hd, scale, window=0, softcap=0.0, fp8=False, spare_blocks=0):
    torch.manual_seed(len(lens) * 1000 + sum(lens) + hd)
    need = [(n + c + 15) // 16 for n, c in zip(lens, ctxs)]
    nb = sum(need) + 1
    order = torch.randperm(nb - 1) + 1
    bt = torch.zeros(len(lens), max(need) + spare_blocks, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = order[at : at + n]
        at += n
    kc = torch.randn(nb, nkv, 16, hd, device=DEV, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    # rows that no query sees must not reach the result
    for i, (n, c) in enumerate(zip(lens, ctxs)):
        if (n + c) % 16:
            kc[bt[i, need[i] - 1], :, (n + c) % 16 :] = float("nan")
            vc[bt[i, need[i] - 1], :, (n + c) % 16 :] = float("nan")
    if fp8:
        kc, vc = kc.to(torch.float8_e5m2), vc.to(torch.float8_e5m2)
    qkv = torch.randn(sum(lens), (nq + 2) * hd, device=DEV, dtype=torch.bfloat16)
    q = qkv[:, : nq * hd].unflatten(-1, (nq, hd))  # strided rows, as in the model
    start = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    total = torch.tensor([n + c for n, c in zip(lens, ctxs)], dtype=torch.int32, device=DEV)
    got = ops.paged_attention_prefill(q, kc, vc, bt.to(DEV), start, total, scale,
                                      window=window, softcap=softcap)
    want = ref.paged_attention_prefill(q.float(), kc.float(), vc.float(), bt.to(DEV), start,
                                       total, scale, window=window, softcap=softcap)
    vmax = torch.nan_to_num(vc.float()).abs().max().item()
    torch.testing.assert_close(got.float(), want, atol=2 * 2.0 ** -9 * vmax, rtol=2 * 2.0 ** -9)


@pytest.mark.parametrize("group", [1, 2, 4, 8])
@pytest.mark.parametrize("hd", [128, 256])
def test_row_and_key_remainders(group, hd):
    _run([1, 31, 32, 33, 65, 127, 128, 129], [0, 1, 32, 63, 64, 65, 15, 200],
         2 * group, 2, hd, hd ** -0.5)


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("window", [1, 31, 64, 65])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_windows(hd, window, softcap):
    _run([3, 100, 40], [130, 0, 64], 4, 2, hd, hd ** -0.5, window=window, softcap=softcap)


@pytest.mark.parametrize("group", [1, 2, 8])
@pytest.mark.parametrize("window", [0, 64, 65, 129, 161, 200, 300])
@pytest.mark.parametrize("softcap,fp8", [(0.0, False), (20.0, False), (0.0, True)])
def test_head_size_256_on_both_sides_of_192_keys(group, window, softcap, fp8):
    """Up to 192 keys a workgroup (a window and the 32 to 128 rows behind it count as its
    most) have a kernel of their own: the same from tables of 12 blocks, and of more."""
    for lens, ctxs in [([64, 3, 33], [128, 189, 0]), ([65, 1], [128, 500]),
                       ([3, 100, 130], [330, 0, 264])]:
        _run(lens, ctxs, 2 * group, 2, 256, 0.07, window=window, softcap=softcap, fp8=fp8)
    _run([40, 17], [0, 3], 2 * group, 2, 256, 0.07, window=window, softcap=softcap, fp8=fp8,
         spare_blocks=13)


@pytest.mark.parametrize("hd", [128, 256])
def test_eight_bit_cache(hd):
    _run([70, 5], [33, 100], 8, 2, hd, hd ** -0.5, fp8=True)


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("spread", [0.2, 0.7, 2.5])
def test_softcap_on_both_sides_of_its_forms(hd, spread):
    """Scores about and on both sides of 0.7 of the cap, where the form changes."""
    _run([70], [33], 4, 2, hd, spread * 20.0 * hd ** -0.5, softcap=20.0)


def test_softcap_small_and_large_scores():
    _run([80], [40], 4, 1, 256, 1e-4, softcap=50.0)
    _run([80], [40], 4, 1, 256, 2.0, softcap=30.0)


def test_negative_and_zero_scale():
    _run([50, 17], [20, 0], 4, 1, 128, -0.05)
    _run([50, 17], [20, 0], 4, 1, 128, 0.0)


def test_wide_block_tables_and_many_short_runs():
    _run([16] * 70 + [200] + [1] * 30, [0] * 70 + [5] + [40] * 30, 8, 2, 128, 0.09,
         spare_blocks=40)


@pytest.mark.parametrize("first,lens", [(100, [200]), (1, [40, 33, 0, 129]), (255, [1, 31, 300])])
def test_runs_of_a_longer_stream(first, lens):
    """Offsets that do not begin at 0: the rows before them are not touched."""
    torch.manual_seed(first)
    nq, nkv, hd, ctx = 8, 2, 128, 20
    need = [(n + ctx + 15) // 16 for n in lens]
    bt = torch.zeros(len(lens), max(need), dtype=torch.int32)
    at = 1
    for i, n in enumerate(need):
        bt[i, :n] = torch.arange(at, at + n)
        at += n
    kc = torch.randn(at, nkv, 16, hd, device=DEV, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    q = torch.randn(first + sum(lens), nq, hd, device=DEV, dtype=torch.bfloat16)
    ends = [first + sum(lens[:i]) for i in range(len(lens) + 1)]
    start = torch.tensor(ends, dtype=torch.int32, device=DEV)
    total = torch.tensor([n + ctx for n in lens], dtype=torch.int32, device=DEV)
    got = torch.full_like(q, 7.0)
    ops.paged_attention_prefill(q, kc, vc, bt.to(DEV), start, total, 0.09, out=got)
    want = ref.paged_attention_prefill(q[first:].float(), kc.float(), vc.float(), bt.to(DEV),
                                       start - first, total, 0.09)
    assert (got[:first] == 7.0).all()
    torch.testing.assert_close(got[first:].float(), want, rtol=2 * 2.0 ** -9,
                               atol=2 * 2.0 ** -9 * vc.float().abs().max().item())


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_keys_that_are_not_finite(hd, softcap):
    """A NaN score reaches the rows that see it; a capped infinite one is the cap."""
    torch.manual_seed(hd)
    kc = torch.randn(10, 1, 16, hd, device=DEV, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    kc[2, 0, 5, 7] = float("nan")
    kc[5, 0, 3, 1], kc[8, 0, 3, 1] = float("inf"), -float("inf")
    bt = torch.tensor([[1, 2, 3], [4, 5, 6], [7, 8, 9]], dtype=torch.int32, device=DEV)
    total = torch.full((3,), 40, dtype=torch.int32, device=DEV)
    start = torch.tensor([0, 40, 80, 120], dtype=torch.int32, device=DEV)
    q = torch.randn(120, 2, hd, device=DEV, dtype=torch.bfloat16)
    args = (bt, start, total, hd ** -0.5)
    got = ops.paged_attention_prefill(q, kc, vc, *args, softcap=softcap).float()
    want = ref.paged_attention_prefill(q.float(), kc.float(), vc.float(), *args, softcap=softcap)
    assert want[21:40].isnan().all() and want[:21].isfinite().all()
    if softcap:
        bound = 2 * 2.0 ** -9 * vc.float().abs().max().item()
        torch.testing.assert_close(got, want, atol=bound, rtol=2 * 2.0 ** -9, equal_nan=True)
    else:  # an infinite score outweighs all others or is outweighed
        assert torch.equal(got.isnan(), want.isnan())


@pytest.mark.parametrize("window", [0, 50, 90])
@pytest.mark.parametrize("n,ctx", [(1, 0), (33, 31), (64, 0), (97, 100), (200, 17), (97, 132),
                                   (170, 251)])
def test_maxima_that_grow_with_every_tile(n, ctx, window):
    """Head size 256, the sums rescaled in most iterations: each key's score is above
    the last one's, by 2^4 a tile of 32 keys. Odd and even numbers of tiles; windows
    that begin behind a wave's first tiles."""
    torch.manual_seed(n)
    total, hd = n + ctx, 256
    kc = torch.zeros((total + 15) // 16 + 1, 2, 16, hd, device=DEV, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    at = torch.arange(total, device=DEV)
    kc[at // 16 + 1, :, at % 16, 0] = (at // 4 * 0.35)[:, None].bfloat16()
    bt = torch.arange(1, kc.shape[0], device=DEV, dtype=torch.int32)[None]
    q = torch.randn(n, 2, hd, device=DEV, dtype=torch.bfloat16)
    q[:, :, 0] = 1.0
    start = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    lens = torch.tensor([total], dtype=torch.int32, device=DEV)
    got = ops.paged_attention_prefill(q, kc, vc, bt, start, lens, 1.0, window=window)
    want = ref.paged_attention_prefill(q.float(), kc.float(), vc.float(), bt, start, lens, 1.0,
                                       window=window)
    torch.testing.assert_close(got.float(), want, rtol=2 * 2.0 ** -9,
                               atol=2 * 2.0 ** -9 * vc.float().abs().max().item())
