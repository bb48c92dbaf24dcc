"""Decode attention over planned splits against the reference, and what a plan holds."""
import random

import pytest
import torch

from kubeai_amd import ops
from kubeai_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
BS = 16


def _caches(lens, n_kv, hd, dtype, seed):
    need = [max(1, -(-n // BS)) for n in lens]
    g = torch.Generator(device=DEV).manual_seed(seed)
    kc, vc = (torch.randn(sum(need) + 1, n_kv, BS, hd, device=DEV, generator=g).to(dtype)
              for _ in range(2))
    ids = list(range(1, sum(need) + 1))
    random.Random(seed).shuffle(ids)
    bt = torch.zeros(len(lens), max(need), dtype=torch.int32)
    for i, n in enumerate(need):
        bt[i, :n] = torch.tensor([ids.pop() for _ in range(n)])
    return kc, vc, bt.to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV)


LENGTHS = {
    "one": [1], "one long": [5003], "one of many": [37] * 9 + [3000] + [200] * 14,
    "edges": [1, 15, 16, 17, 31, 32, 33, 127, 128, 129, 255, 256, 257, 2048, 2049],
    "even": [512] * 32, "many": [1 + 7 * i % 400 for i in range(130)],
}


@pytest.mark.parametrize("lens", LENGTHS.values(), ids=LENGTHS.keys())
@pytest.mark.parametrize("n_kv,tile,window", [(8, 16, 0), (1, 32, 0), (4, 16, 100), (300, 16, 0)])
def test_plan_names_every_split_once(lens, n_kv, tile, window):
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    plan = ops._C.paged_decode_plan(sl, n_kv, 128, 2 if tile == 16 else 1, window).cpu()
    B, M = len(lens), max(1, 256 // n_kv)
    n = 3 * M + B
    items, rows = plan[: 4 * n].view(n, 4).tolist(), plan[4 * n :].view(B, 2).tolist()
    used = sum(k for _, k in rows)
    assert sorted(i for at, k in rows for i in range(at, at + k)) == list(range(used))
    got = {}
    for row, length, packed, part in items[:used]:
        split, splits = packed & 0xFFFF, packed >> 16
        at, k = rows[row]
        assert length == lens[row] and splits == k and part == at + split and 0 <= split < k
        got.setdefault(row, set()).add(split)
    assert all(got[i] == set(range(rows[i][1])) for i in range(B))
    assert all(it[0] == -1 for it in items[used:])
    assert all(1 <= k <= 16 for _, k in rows)


@pytest.mark.parametrize("lens", LENGTHS.values(), ids=LENGTHS.keys())
@pytest.mark.parametrize("n_q,n_kv,hd,dtype,window,cap", [
    (32, 8, 128, torch.bfloat16, 0, 0.0),
    (8, 1, 128, torch.float8_e5m2, 0, 0.0),
    (8, 4, 256, torch.bfloat16, 100, 30.0),
    (40, 8, 128, torch.bfloat16, 700, 0.0),
])
def test_planned_attention(lens, n_q, n_kv, hd, dtype, window, cap):
    kc, vc, bt, sl = _caches(lens, n_kv, hd, dtype, n_q + len(lens))
    q = torch.randn(len(lens), n_q, hd, device=DEV).bfloat16()
    plans = {}
    plan = ops.decode_plan(plans, sl, bt, kc, window)
    assert ops.decode_plan(plans, sl, bt, kc, window) is plan  # one a step
    kw = dict(window=window, softcap=cap)
    got = ops.paged_attention_decode(q, kc, vc, bt, sl, hd**-0.5, plan=plan, **kw)
    want = ref.paged_attention_decode(q.float(), kc.float(), vc.float(), bt, sl, hd**-0.5, **kw)
    # rounded once to bf16 (half a unit, 2^-9), fp32 within
    err = (got.float() - want).abs()
    assert torch.all(err <= 2.0**-8 * want.abs() + 1e-4)
    f8, scale = ops.paged_attention_decode_fp8(q, kc, vc, bt, sl, hd**-0.5, plan=plan, **kw)
    w8, wscale = ops.quant_fp8(got.view(len(lens), -1))
    assert torch.equal(f8.view(torch.uint8), w8.view(torch.uint8))
    assert torch.equal(scale, wscale.view(-1))


def test_no_plan():
    kc, vc, bt, sl = _caches([20, 30], 2, 128, torch.bfloat16, 0)
    assert ops.decode_plan(None, sl, bt, kc) is None
    assert ops.decode_plan({}, sl.cpu(), bt.cpu(), kc) is None
    assert ops.decode_plan({}, sl.expand(600, 2).reshape(-1), bt, kc) is None


def test_a_recorded_plan_follows_the_lengths():
    kc, vc, bt, sl = _caches([700, 90, 333], 8, 128, torch.bfloat16, 1)
    q = torch.randn(3, 32, 128, device=DEV).bfloat16()

    def step():
        plan = ops.decode_plan({}, sl, bt, kc)
        return ops.paged_attention_decode(q, kc, vc, bt, sl, 0.1, plan=plan)

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for lens in ([700, 90, 333], [1, 80, 5], [650, 1, 320], [16, 17, 200]):
        sl.copy_(torch.tensor(lens, dtype=torch.int32))
        graph.replay()
        want = ref.paged_attention_decode(q.float(), kc.float(), vc.float(), bt, sl, 0.1)
        assert torch.all((out.float() - want).abs() <= 2.0**-8 * want.abs() + 1e-4)


@pytest.mark.parametrize("planned", [True, False])
@pytest.mark.parametrize("lens", [LENGTHS[k] for k in ("one", "one long", "edges", "even")],
                         ids=["one", "one long", "edges", "even"])
@pytest.mark.parametrize("n_q,n_kv,hd,window,cap,parts,scaled", [
    (32, 8, 128, 0, 0.0, 4, True),
    (8, 1, 128, 0, 0.0, 7, False),
    (8, 4, 256, 100, 30.0, 1, True),
    (12, 2, 256, 0, 0.0, 8, False),
    (2, 2, 128, 33, 20.0, 3, True),
])
def test_from_sums(lens, n_q, n_kv, hd, window, cap, parts, scaled, planned):
    """One launch against rotation, cache write and attention after one another: the
    same bits in the caches (angles are powers of 2: a product is exact, so it does not
    matter which of two the compiler fuses with the sum), and results that differ by a
    rounding here and there (sums in fp32 may be fused differently, 2^-24 of them, which is
    the other side of a rounding to 2^-9 once in some ten thousand). A row without a slot
    keeps its key from the cache."""
    B, width = len(lens), (n_q + 2 * n_kv) * hd
    kc, vc, bt, sl = _caches(lens, n_kv, hd, torch.bfloat16, parts)
    g = torch.Generator(device=DEV).manual_seed(7)
    part = torch.randn(parts, B, width, device=DEV, generator=g) * parts**-0.5
    scales = (torch.rand(B, device=DEV) + 0.5, torch.rand(width, device=DEV) + 0.5)
    qkv = ops.ProductSums(part, *(scales if scaled else (None, None)))
    pos = sl - 1
    angle = pos.max().item() + 1
    cos_sin = 2.0 ** -torch.randint(0, 4, (angle, hd), device=DEV, generator=g).float()
    cos_sin[:, ::3] *= -1.0
    at = (sl - 1).long()
    slots = bt.gather(1, (at // BS)[:, None]).long()[:, 0] * BS + at % BS
    if B > 2:
        slots[1] = -1
    plan = ops.decode_plan({}, sl, bt, kc, window) if planned else None
    one, two = (kc.clone(), vc.clone()), (kc.clone(), vc.clone())
    q = ops.rope_and_cache(qkv, n_q, pos, cos_sin, *one, slots)
    kw = dict(window=window, softcap=cap, plan=plan)
    want = ops.paged_attention_decode(q, *one, bt, sl, hd**-0.5, **kw)
    assert ops.decode_takes_sums(qkv, n_q, cos_sin, *two)
    got = ops.paged_attention_decode_sums(qkv, n_q, pos, cos_sin, slots, *two, bt, sl,
                                          hd**-0.5, **kw)
    assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1])
    diff = (got.float() - want.float()).abs()
    assert torch.all(diff <= 2.0**-7 * want.float().abs() + 2.0**-21)
    assert (diff > 0).float().mean() < 2e-3
    two = (kc.clone(), vc.clone())
    f8, scale = ops.paged_attention_decode_sums(qkv, n_q, pos, cos_sin, slots, *two, bt, sl,
                                                hd**-0.5, fp8=True, **kw)
    w8, wscale = ops.quant_fp8(got.view(B, -1))
    assert torch.equal(f8.view(torch.uint8), w8.view(torch.uint8))
    assert torch.equal(scale.view(-1), wscale.view(-1))
    assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1])


@pytest.mark.parametrize("planned_rows", [1, 7, 9, 40])
def test_plans_of_other_rows_are_refused(planned_rows):
    """Their numbers would be taken as rows of q and as parts: nothing is launched."""
    kc, vc, bt, sl = _caches([30] * 40, 8, 128, torch.bfloat16, 0)
    plan = ops.decode_plan({}, sl[:planned_rows].contiguous(), bt, kc)
    q = torch.randn(9, 32, 128, device=DEV).bfloat16()
    caches = (kc, vc, bt[:8].contiguous(), sl[:8].contiguous())
    own = ops.decode_plan({}, caches[3], bt, kc)
    prompt = (bt[8:9].contiguous(), torch.tensor([0, 1], dtype=torch.int32, device=DEV),
              sl[8:9].contiguous())
    ops.paged_attention_decode(q[:8], *caches, 0.1, plan=own)
    ops.paged_attention_step(q, 8, *caches, *prompt, 0.1, plan=own)
    for wrong in (plan, own[:-1], own[:-6], torch.cat([own, own[:6]])):
        with pytest.raises(RuntimeError, match="a plan of 8 rows"):
            ops.paged_attention_decode(q[:8], *caches, 0.1, plan=wrong)
        with pytest.raises(RuntimeError, match="a plan of 8 rows"):
            ops.paged_attention_step(q, 8, *caches, *prompt, 0.1, plan=wrong)
    # of other kv heads than the cache's
    other = ops._C.paged_decode_plan(caches[3], 4, 128, 2, 0)
    with pytest.raises(RuntimeError, match="over 8 kv heads"):
        ops.paged_attention_decode(q[:8], *caches, 0.1, plan=other)


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("planned", [True, False])
def test_rows_of_no_keys_need_no_table(planned, hd):
    """As with a table whose entries do not count: no number, and nothing read for it."""
    kc, vc, _, _ = _caches([30], 4, hd, torch.bfloat16, 0)
    sl = torch.zeros(3, dtype=torch.int32, device=DEV)
    q = torch.randn(4, 8, hd, device=DEV).bfloat16()
    prompt = (torch.zeros(1, 1, dtype=torch.int32, device=DEV),
              torch.tensor([0, 1], dtype=torch.int32, device=DEV), sl[:1] + 1)
    for columns in (1, 0):
        bt = torch.zeros(3, columns, dtype=torch.int32, device=DEV)
        plan = ops.decode_plan({}, sl, bt, kc) if planned else None
        got = ops.paged_attention_decode(q[:3], kc, vc, bt, sl, 0.1, plan=plan)
        assert got.isnan().all()
        if planned and hd == 128:
            got = ops.paged_attention_step(q, 3, kc, vc, bt, sl, *prompt, 0.1, plan=plan)
            assert got[:3].isnan().all() and not got[3:].isnan().any()


@pytest.mark.parametrize("n_q,n_kv", [(16, 4), (20, 4), (32, 8)])
@pytest.mark.parametrize("lens", [LENGTHS[k] for k in ("one long", "one of many", "edges")],
                         ids=["one long", "one of many", "edges"])
def test_heads_of_256_to_eight_bits(lens, n_q, n_kv):
    """One wave merges one head, or two of which the second may not be there, in up to 16
    splits: the bits of the merge and the conversion after one another."""
    kc, vc, bt, sl = _caches(lens, n_kv, 256, torch.bfloat16, n_q)
    q = torch.randn(len(lens), n_q, 256, device=DEV).bfloat16()
    plan = ops.decode_plan({}, sl, bt, kc)
    want = ops.paged_attention_decode(q, kc, vc, bt, sl, 0.06, plan=plan)
    f8, scale = ops.paged_attention_decode_fp8(q, kc, vc, bt, sl, 0.06, plan=plan)
    w8, wscale = ops.quant_fp8(want.view(len(lens), -1))
    assert torch.equal(f8.view(torch.uint8), w8.view(torch.uint8))
    assert torch.equal(scale, wscale.view(-1))


@pytest.mark.parametrize("rows,columns,n_kv,window,alone,planned", [
    (8, 8, 8, 0, True, False), (8, 9, 8, 0, True, True), (9, 8, 8, 0, True, True),
    (64, 8, 8, 0, True, False), (64, 9, 8, 0, True, True), (64, 8, 8, 0, False, True),
    (1, 1, 8, 0, True, False), (1, 2, 8, 0, True, False), (1, 512, 8, 0, True, True),
    (64, 512, 8, 128, True, False), (64, 512, 8, 129, True, True),
    (256, 9, 1, 0, True, True), (257, 512, 1, 0, True, False), (257, 512, 1, 0, False, True),
    (512, 512, 8, 0, False, True), (513, 512, 8, 0, False, False),
])
def test_where_rows_are_planned(rows, columns, n_kv, window, alone, planned):
    cache = torch.empty(1, n_kv, BS, 128, dtype=torch.bfloat16, device=DEV)
    sl = torch.ones(rows, dtype=torch.int32, device=DEV)
    bt = torch.zeros(rows, columns, dtype=torch.int32, device=DEV)
    plan = ops.decode_plan({}, sl, bt, cache, window, alone=alone)
    assert (plan is not None) is planned
    assert ops.decode_plan(None, sl, bt, cache, window, alone=alone) is None


@pytest.mark.parametrize("columns", [1, 4, 5, 8, 9])
@pytest.mark.parametrize("rows,n_kv,window,cap", [(70, 8, 0, 0.0), (3, 2, 0, 20.0), (70, 8, 50, 0.0)])
def test_one_tile_a_wave(rows, columns, n_kv, window, cap):
    """Without a plan: tiles of one block, of two where a wave then has one, and a loop."""
    g = random.Random(columns)
    lens = [16 * columns - g.randrange(16 * columns) for _ in range(rows)]
    lens[0] = 16 * columns
    kc, vc, bt, sl = _caches(lens, n_kv, 128, torch.bfloat16, columns)
    q = torch.randn(rows, 4 * n_kv, 128, device=DEV).bfloat16()
    kw = dict(window=window, softcap=cap)
    got = ops.paged_attention_decode(q, kc, vc, bt, sl, 0.09, **kw)
    want = ref.paged_attention_decode(q.float(), kc.float(), vc.float(), bt, sl, 0.09, **kw)
    assert torch.all((got.float() - want).abs() <= 2.0**-8 * want.abs() + 1e-4)
