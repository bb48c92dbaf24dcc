"""A row whose logits hold no number ends its own request and no other one."""
import math

import pytest
import torch
from fastapi.testclient import TestClient

from kubeai_amd import ops
from kubeai_amd.engine import EngineConfig, LLMEngine, SamplingParams
from kubeai_amd.engine.server import EngineServer, build_app


def _engine():
    return LLMEngine(EngineConfig(model="llama-tiny", device="cpu", num_gpu_blocks=64,
                                  max_model_len=256, max_num_seqs=8))


def _run(eng, requests):
    for rid, params in requests.items():
        eng.add_request(list(range(10, 30)), params, request_id=rid)
    seen, last = {rid: [] for rid in requests}, {}
    for _ in range(40):
        if not eng.has_work():
            break
        for o in eng.step():
            seen[o.request_id] += o.new_token_ids
            last[o.request_id] = o
    assert not eng.has_work()
    return seen, last


def _behind_the_vocabulary(monkeypatch, which):
    """The samplers as they are on the GPU: a row in which no value compares gives the
    number behind the vocabulary (on the CPU argmax gives the first NaN's place)."""
    real_block, real_gumbel = ops.sample_with_logprobs, ops.gumbel_sample

    def behind(logits, tokens):
        bad = logits.isnan().all(-1)
        which.append(int(bad.sum()))
        return torch.where(bad, logits.shape[1], tokens)

    def block(logits, *args):
        got = real_block(logits, *args)
        tokens = got[: 8 * len(logits)].view(torch.int64)
        tokens.copy_(behind(logits, tokens))
        return got

    monkeypatch.setattr(ops, "sample_with_logprobs", block)
    monkeypatch.setattr(ops, "gumbel_sample",
                        lambda logits, *a: behind(logits, real_gumbel(logits, *a)))
    # (the CPU's form of the test for membership reads the candidate's logit)
    real_accept = ops.nucleus_accept
    monkeypatch.setattr(ops, "nucleus_accept", lambda lg, cand, *a: real_accept(
        lg, cand.clamp_max(lg.shape[1] - 1), *a))


@pytest.mark.parametrize("good", [
    {}, {"temperature": 0.8, "seed": 3}, {"temperature": 0.8, "seed": 3, "top_p": 0.9},
    {"logprobs": 2}, {"json_mode": True},
])
def test_other_requests_go_on(monkeypatch, good):
    params = dict(max_tokens=6, ignore_eos=True)
    alone, _ = _run(_engine(), {"good": SamplingParams(**params, **good)})
    which = []
    _behind_the_vocabulary(monkeypatch, which)
    eng = _engine()
    # from the second token on its penalty makes every logit NaN
    bad = SamplingParams(**params, frequency_penalty=math.nan, **good)
    free = eng.block_manager.usage()
    seen, last = _run(eng, {"good": SamplingParams(**params, **good), "bad": bad})
    assert max(which) == 1
    assert seen["good"] == alone["good"] and last["good"].finish_reason == "length"
    assert len(seen["bad"]) == 1 and last["bad"].finish_reason == "abort"
    assert last["bad"].new_token_ids == [] and last["bad"].logprob is None
    assert last["bad"].top_logprobs is None and last["bad"].output_token_ids == seen["bad"]
    assert not eng.scheduler.running
    assert eng.block_manager.usage() == free


@pytest.fixture(scope="module")
def client():
    server = EngineServer(EngineConfig(model="llama-tiny", device="cpu", num_gpu_blocks=64,
                                       max_model_len=256), "m")
    server.start()
    server._ready.wait(timeout=60)
    with TestClient(build_app(server)) as c:
        yield c
    server.stop()


@pytest.mark.parametrize("body", [
    {"temperature": "nan"}, {"top_p": "NaN"}, {"presence_penalty": "inf"},
    {"frequency_penalty": "-inf"}, {"frequency_penalty": "nan"},
    {"frequency_penalty": 4e38},  # infinite in 32 bits
])
def test_numbers_that_are_none_are_refused(client, body):
    r = client.post("/v1/completions", json={"prompt": "a b", "max_tokens": 2, **body})
    assert r.status_code == 400 and next(iter(body)) in r.json()["error"]["message"]


@pytest.mark.parametrize("body", [
    {"temperature": "inf"}, {"top_p": "inf"}, {"temperature": "-inf"}, {"top_p": ""},
    {"presence_penalty": 3e38, "temperature": 0},
])
def test_what_was_taken_is_taken(client, body):
    r = client.post("/v1/completions", json={"prompt": "a b", "max_tokens": 2, **body})
    assert r.status_code == 200


@pytest.mark.gpu
@pytest.mark.parametrize("V", [1, 1000, 4099])
def test_candidates_outside_the_vocabulary(V):
    """None is in the nucleus, and no logit is read for it (the last row's would lie
    behind them all); the row beside it draws what it draws alone."""
    from kubeai_amd.engine.runner import _sample_topk_topp

    x = torch.randn(2, V, device="cuda")
    x[1] = float("nan")
    temps = torch.ones(2, device="cuda")
    m, z = ops.nucleus_stats(x, temps)
    top_p = torch.full((2,), 0.9, device="cuda")
    top_k = torch.zeros(2, dtype=torch.int32, device="cuda")
    best = x[0].argmax().item()
    for none in (V, -1):
        cand = torch.tensor([best, none], device="cuda")
        ok = ops.nucleus_accept(x, cand, m, z, temps, top_p, top_k)
        assert ok.tolist() == [1, 0]
    seeds = torch.tensor([4, 5], device="cuda")
    both = _sample_topk_topp(x, [0.9] * 2, [0] * 2, [1.0] * 2, temps, seeds, 3)
    one = _sample_topk_topp(x[:1], [0.9], [0], [1.0], temps[:1], seeds[:1], 3)
    assert both.tolist() == [one.item(), V]
