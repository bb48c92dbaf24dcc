"""A step's prompt portions and decode rows in one launch: the bits of the two launches,
whose results are tested against the oracle, and the oracle itself."""
import math

import pytest
import torch

from kubeai_amd import ops
from kubeai_amd.ops import ref

pytestmark = pytest.mark.gpu

STEPS = [  # lengths of decode rows, (cached, new) tokens of prompts
    ([1], [(0, 1)]),
    ([16, 17], [(0, 32), (15, 33)]),
    ([700, 5, 300], [(600, 112), (0, 1), (0, 1), (64, 64)]),  # padding runs among them
    ([40] * 40, [(0, 17)]),
    ([3000, 20], [(300, 129)]),
    ([30] * 3, [(0, 1021)]),  # 1024 rows
    ([30] * 4, [(0, 1021)]),
]


def _step(dec, seqs, heads, kv_heads, dtype):
    g = torch.Generator().manual_seed(len(dec) + heads)
    need = [-(-n // 16) for n in dec] + [-(-(c + n) // 16) for c, n in seqs]
    ids = (torch.randperm(sum(need), generator=g) + 1).int().split(need)

    def table(rows):
        t = torch.zeros(len(rows), max(len(r) for r in rows) + 1, dtype=torch.int32)
        for i, r in enumerate(rows):
            t[i, : len(r)] = r
        return t.cuda()

    T = len(dec) + sum(n for _, n in seqs)
    # rows of q lie apart, as in a product's q | k | v
    q = torch.randn(T, heads + 2 * kv_heads, 128, generator=g).bfloat16().cuda()[:, :heads]
    shape = (sum(need) + 1, kv_heads, 16, 128)
    caches = [torch.randn(shape, generator=g).to(dtype).cuda() for _ in range(2)]
    start = torch.tensor([0] + [n for _, n in seqs]).cumsum(0).int().cuda()
    return dict(
        q=q, caches=caches, dec=(table(ids[: len(dec)]), torch.tensor(dec).int().cuda()),
        pre=(table(ids[len(dec) :]), start,
             torch.tensor([c + n for c, n in seqs]).int().cuda()))


@pytest.mark.parametrize("dec,seqs", STEPS)
@pytest.mark.parametrize("heads,kv_heads", [(32, 8), (4, 4), (8, 4), (64, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e5m2])
@pytest.mark.parametrize("window,softcap", [(0, 0.0), (37, 0.0), (0, 20.0), (100, 5.0)])
def test_step_is_its_two_halves(dec, seqs, heads, kv_heads, dtype, window, softcap):
    s, nd, scale = _step(dec, seqs, heads, kv_heads, dtype), len(dec), 1 / math.sqrt(128)
    kw = dict(window=window, softcap=softcap)
    plan = ops.decode_plan({}, s["dec"][1], s["dec"][0], s["caches"][0], window)
    assert ops.step_attention_takes(s["q"], nd, s["caches"][0], plan)
    want = torch.empty(s["q"].shape, dtype=torch.bfloat16, device="cuda")
    ops.paged_attention_decode(s["q"][:nd], *s["caches"], *s["dec"], scale, out=want[:nd],
                               plan=plan, **kw)
    ops.paged_attention_prefill(s["q"][nd:], *s["caches"], *s["pre"], scale, out=want[nd:], **kw)
    args = (s["q"], nd, *s["caches"], *s["dec"], *s["pre"], scale)
    assert torch.equal(ops.paged_attention_step(*args, plan=plan, **kw), want)
    got, by = ops.paged_attention_step(*args, plan=plan, fp8=True, **kw)
    rows, row_scale = ops.quant_fp8(want.view(len(want), -1))
    assert torch.equal(got.view(torch.uint8), rows.view(torch.uint8))
    assert torch.equal(by, row_scale)


@pytest.mark.parametrize("window,softcap", [(0, 0.0), (37, 20.0)])
def test_step_against_the_oracle(window, softcap):
    dec, seqs = STEPS[2]
    s, nd, scale = _step(dec, seqs, 8, 2, torch.bfloat16), len(dec), 1 / math.sqrt(128)
    kw = dict(window=window, softcap=softcap)
    plan = ops.decode_plan({}, s["dec"][1], s["dec"][0], s["caches"][0], window)
    got = ops.paged_attention_step(s["q"], nd, *s["caches"], *s["dec"], *s["pre"], scale,
                                   plan=plan, **kw).float()
    caches = [c.float() for c in s["caches"]]
    want = torch.cat([
        ref.paged_attention_decode(s["q"][:nd].float(), *caches, *s["dec"], scale, **kw),
        ref.paged_attention_prefill(s["q"][nd:].float(), *caches, *s["pre"], scale, **kw)])
    # the result's and the prompts' weights' rounding to bf16: 2^-9 each, at most
    assert (got - want).norm() / want.norm() < 4e-3


def test_steps_that_are_not_taken():
    s = _step([30], [(0, 20)], 8, 4, torch.bfloat16)
    plan = ops.decode_plan({}, s["dec"][1], s["dec"][0], s["caches"][0])
    takes = ops.step_attention_takes
    assert not takes(s["q"], 1, s["caches"][0], None)
    assert not takes(s["q"], 0, s["caches"][0], plan)
    assert not takes(s["q"][:1], 1, s["caches"][0], plan)
    assert not takes(s["q"][..., :64], 1, s["caches"][0], plan)
    assert not takes(s["q"][:, :6], 1, s["caches"][0], plan)
