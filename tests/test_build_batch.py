"""The tensors of a step (ModelRunner.build_batch) against plain lists: decode
rows, prompt portions shorter and longer than a cache block, padding to a step
size, adapters, state slots; on a GPU they are views of one copy."""
import random

import pytest
import torch

from kubeai_amd.engine import EngineConfig, LLMEngine, SamplingParams
from kubeai_amd.engine.runner import _bucket
from kubeai_amd.engine.scheduler import Request, ScheduledSeq, SchedulerOutput

BLOCK = 16


def _engine(model, device):
    return LLMEngine(EngineConfig(
        model=model, device=device, num_gpu_blocks=64, max_model_len=512, max_num_seqs=16,
        max_num_batched_tokens=512, enable_prefix_caching=False))


def _step(rng, rows, portions, adapters):
    seqs = []
    for i, (c, n) in enumerate([(rng.randrange(0, 200), 1) for _ in range(rows)] + portions):
        r = Request([rng.randrange(3, 99) for _ in range(c + n)], SamplingParams(),
                    request_id="r%d" % i, lora_id=i % 3 if adapters else 0)
        r.block_table = [rng.randrange(1, 64) for _ in range((c + n + BLOCK - 1) // BLOCK)]
        r.state_slot = i
        seqs.append(ScheduledSeq(r, c, n))
    return SchedulerOutput(decode=seqs[:rows], prefill=seqs[rows:], preempted=[])


def _check(runner, out, want=None):
    fb = runner.build_batch(out, want=want)
    ids, pos, slots, lora, lens, starts, tables = [], [], [], [], [], [0], []
    for ss in out.all_seqs:
        for i in range(ss.chunk_start, ss.chunk_start + ss.chunk_len):
            ids.append(ss.req.tokens[i])
            pos.append(i)
            slots.append(ss.req.block_table[i // BLOCK] * BLOCK + i % BLOCK)
            lora.append(ss.req.lora_id)
        lens.append(ss.chunk_start + ss.chunk_len)
        starts.append(len(ids))
        tables.append(ss.req.block_table)
    state = [ss.req.state_slot for ss in out.all_seqs]
    while len(ids) < _bucket(starts[len(out.all_seqs)]):
        n = min(BLOCK, _bucket(starts[len(out.all_seqs)]) - len(ids))
        ids, pos, slots = ids + [0] * n, pos + list(range(n)), slots + [-1] * n
        lora, lens, tables, state = lora + [0] * n, lens + [n], tables + [[]], state + [-1]
        starts.append(len(ids))
    width = max([len(t) for t in tables] + [1])
    tables = [t + [0] * (width - len(t)) for t in tables]
    nd = len(out.decode)

    def same(t, values, dtype=torch.int32):
        assert t.dtype == dtype and t.device.type == runner.device.type and t.is_contiguous()
        assert t.tolist() == values

    same(fb.input_ids, ids)
    same(fb.positions, pos)
    same(fb.slot_mapping, slots, torch.int64)
    assert fb.n_decode == nd and fb.n_prefill == len(lens) - nd
    if nd:
        same(fb.decode_block_tables, tables[:nd])
        same(fb.decode_seq_lens, lens[:nd])
    else:
        assert fb.decode_block_tables is None and fb.decode_seq_lens is None
    if fb.n_prefill:
        same(fb.prefill_block_tables, tables[nd:])
        same(fb.prefill_seq_lens, lens[nd:])
        same(fb.prefill_query_start_loc, [s - nd for s in starts[nd:]])
    else:
        assert fb.prefill_block_tables is None and fb.prefill_query_start_loc is None
    if want is None:
        rows = list(range(nd)) + [starts[i + 1] - 1 for i in range(nd, len(out.all_seqs))
                                  if out.all_seqs[i].samples]
    else:
        rows = [starts[i] + o for i, ss in enumerate(out.all_seqs)
                for o in want.get(ss.req.request_id, ())]
    same(fb.logits_indices, rows, torch.int64)
    if runner.lora_manager is not None and runner.lora_manager.active:
        same(fb.lora_ids, lora)
    else:
        assert fb.lora_ids is None
    if runner.uses_seq_meta:
        same(fb.seq.start_loc, starts)
        same(fb.seq.slots, state)
        same(fb.seq.block_tables, tables)
        runs = [b - a for a, b in zip(starts, starts[1:])]
        same(fb.seq.token_seq, [i for i, n in enumerate(runs) for _ in range(n)])
        assert fb.seq.max_len == max(runs) and fb.seq.n_seq == len(runs)
    else:
        assert fb.seq is None


STEPS = [(3, []), (8, []), (0, [(0, 1)]), (0, [(0, 5), (40, 70)]), (5, [(16, 15), (0, 200)]),
         (2, [(7, 64), (100, 65), (3, 2)])]


def _all(model, device, adapters):
    eng = _engine(model, device)
    if adapters:
        eng.load_lora(1, None)
        eng.load_lora(2, None)
    elif not hasattr(eng.runner, "lora_manager"):
        eng.runner.lora_manager = None
    rng = random.Random(5)
    for rows, portions in STEPS:
        out = _step(rng, rows, portions, adapters)
        _check(eng.runner, out)
        _check(eng.runner, out, {"r0": [0], "r1": [0, 0]})


@pytest.mark.parametrize("model,adapters", [("llama-tiny", False), ("llama-tiny", True), ("nugopel-tiny", False)])
def test_step_tensors(model, adapters):
    _all(model, "cpu", adapters)


@pytest.mark.gpu
@pytest.mark.parametrize("model,adapters", [("llama-tiny", False), ("llama-tiny", True), ("nugopel-tiny", False)])
def test_step_tensors_on_the_gpu(model, adapters):
    _all(model, "cuda", adapters)


@pytest.mark.gpu
def test_steps_do_not_share_what_is_still_copied():
    """Many steps are built while the GPU is busy; each keeps its own values."""
    eng = _engine("llama-tiny", "cuda")
    a = torch.randn(4096, 4096, device="cuda")
    for _ in range(20):
        a = torch.tanh(a @ a * 0.01)
    rng, kept = random.Random(6), []
    for i in range(50):
        out = _step(rng, 1 + i % 8, [(0, 30)], False)
        kept.append((eng.runner.build_batch(out), [t for ss in out.all_seqs for t in
                     ss.req.tokens[ss.chunk_start : ss.chunk_start + ss.chunk_len]]))
    for fb, ids in kept:
        assert fb.input_ids[: len(ids)].tolist() == ids


def _runner(hidden, ff, heads, kv_heads, preset="llama-3-8b", shards=1, **other):
    """A runner over an eight-bit model of these widths, without memory for it."""
    import dataclasses

    from kubeai_amd.engine.quant import convert_to_fp8
    from kubeai_amd.engine.runner import ModelRunner
    from kubeai_amd.models.config import PRESETS
    from kubeai_amd.models.llama import LlamaForCausalLM

    # a shard of a tensor-parallel model has a part of the heads and of the inner width
    cfg = dataclasses.replace(
        PRESETS[preset], hidden_size=hidden, intermediate_size=ff // shards,
        num_attention_heads=heads // shards, num_key_value_heads=kv_heads // shards,
        num_hidden_layers=2, vocab_size=64, **other)
    runner = ModelRunner.__new__(ModelRunner)
    runner.model = LlamaForCausalLM(cfg, device="meta")
    convert_to_fp8(runner.model)
    return runner


@pytest.mark.parametrize("n,size", [(256, 256), (257, 272), (546, 560), (1025, 1040), (5174, 5184),
                                    (16384, 16384), (20001, 20001), (40, 40), (97, 128)])
def test_sizes_of_steps_in_eight_bits(n, size):
    """Where all products of a step's rows are the tiled kernel's, steps of more than
    256 tokens are filled up to whole cache blocks."""
    runner = _runner(4096, 14336, 32, 8)
    assert runner._step_size(n) == size
    # a layer that is not in eight bits keeps the sizes of the library
    del runner.model.layers[1]._fp8_widths
    assert runner._step_size(n) == _bucket(n)


@pytest.mark.parametrize("n", [272, 320, 546, 700, 1025, 2000, 3088, 5174, 16000])
@pytest.mark.parametrize("widths", [
    dict(hidden=1536, ff=8960, heads=12, kv_heads=2),              # K below 2048
    dict(hidden=896, ff=4864, heads=7, kv_heads=1),
    dict(hidden=4096, ff=14336, heads=32, kv_heads=8, shards=4),   # o_proj: K 1024
    dict(hidden=4096, ff=14336, heads=32, kv_heads=8, shards=8),
    dict(hidden=4096, ff=14336, heads=32, kv_heads=8, attention_bias=True),
    # (experts on a device where they are not multiplied in one launch)
    dict(hidden=4096, ff=256, heads=32, kv_heads=8, preset="mixtral-8x7b"),
])
def test_steps_with_products_of_the_library_keep_its_sizes(n, widths):
    assert _runner(**widths)._step_size(n) == _bucket(n)


@pytest.mark.parametrize("n,size", [(272, 320), (570, 640), (609, 624), (642, 656), (1030, 1040)])
def test_step_sizes_go_by_the_products_of_their_rows(n, size):
    """2048 x 2048 is the tiled kernel's from 160 tiles of 64 x 128 on: 577 rows."""
    from kubeai_amd import ops

    runner = _runner(2048, 8192, 16, 8)
    assert runner._step_size(n) == size
    assert ops.fp8_product_tiled(577, 2048, 2048) and not ops.fp8_product_tiled(576, 2048, 2048)
    for off in ((600, 2056, 2048), (600, 2048, 2080)):
        assert not ops.fp8_product_tiled(*off)


@pytest.mark.gpu
def test_experts_in_one_launch_are_no_products_of_the_library():
    import dataclasses

    from kubeai_amd.engine.quant import convert_to_fp8
    from kubeai_amd.models.config import PRESETS
    from kubeai_amd.models.llama import LlamaForCausalLM

    for experts, here in ((4, True), (40, False)):  # (40: routed by the library)
        cfg = dataclasses.replace(PRESETS["mixtral-tiny"], num_local_experts=experts)
        model = LlamaForCausalLM(cfg, device="cuda")
        layer = model.layers[0]
        assert not layer.mlp.sorts_here()  # bf16: by the rows
        convert_to_fp8(model)
        assert layer.mlp.sorts_here() is here
        assert layer._fp8_widths == (((512, 256), (256, 256)) if here else None)
