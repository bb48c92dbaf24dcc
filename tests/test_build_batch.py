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


@pytest.mark.parametrize("n,size", [(256, 256), (257, 272), (546, 560), (1025, 1040), (5174, 5184),
                                    (16384, 16384), (20001, 20001), (40, 40), (97, 128)])
def test_sizes_of_steps_in_eight_bits(n, size):
    """Models of eight-bit products fill steps of more than 256 tokens up to whole
    cache blocks; a layer that is not fused keeps the sizes of the library."""
    from kubeai_amd.engine.runner import ModelRunner

    class Any:
        pass

    runner, layers = ModelRunner.__new__(ModelRunner), [Any(), Any()]
    runner.model = Any()
    assert runner._step_size(n) == _bucket(n)
    runner.model.layers = layers
    layers[0]._fp8_fused = True
    assert runner._step_size(n) == _bucket(n)
    layers[1]._fp8_fused = True
    assert runner._step_size(n) == size
