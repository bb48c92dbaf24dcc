"""The serving work that speed is measured on.

Every case is a step, or a short run of steps, that the server's loop makes
all day: a batch of one-token decode rows, a batch of prompt portions (alone
or beside decode rows), or whole requests through `LLMEngine.step`. Widths,
head counts and vocabularies are those of the presets the framework serves
(Llama-3 8B, Mixtral 8x7B, Gemma-2 2B, Nugopel at width 2048); the stacks are
cut to a quarter of their depth or less so that a case can be set up in a
second: every layer does the same work, so times scale with depth.

Decode rows run as the engine runs them, the forward recorded once in a HIP
graph and replayed; prompt portions and steps with adapters go through
`ModelRunner.forward_logits`, the engine's eager step with its batch building.
"""
from __future__ import annotations

import dataclasses
import math
import random
import zlib

import torch

from kubeai_amd.engine import EngineConfig, LLMEngine, SamplingParams
from kubeai_amd.engine.quant import convert_to_fp8
from kubeai_amd.engine.scheduler import Request, ScheduledSeq, SchedulerOutput
from kubeai_amd.models.config import PRESETS

BLOCK = 16  # tokens in a cache block
FAMILIES = {  # preset -> layers kept
    "llama-3-8b": 8, "mixtral-8x7b": 4, "gemma2-2b": 8, "nugopel-2k": 8,
}
RANK = 16  # of the adapters that load_lora makes when it is given no files


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # whole requests: 40 users send a turn of a chat and read a short answer
        # (the scheduler, graph replays and greedy sampling are in it)
        dict(name="chat turn, 40 users", kind="chat", model="llama-3-8b", quant=True,
             rows=40, lo=64, hi=160, new=8),
        # the decode step of that load: 40 rows, a few hundred tokens of history
        dict(name="decode 40 rows fp8", kind="decode", model="llama-3-8b", quant=True,
             rows=40, lo=100, hi=700),
        # one stream on its own, the latency a single user sees
        dict(name="decode 1 row bf16", kind="decode", model="llama-3-8b", quant=False,
             rows=1, lo=3000, hi=3000),
        # a full batch with long histories: cached keys and values outweigh weights
        dict(name="decode 96 rows long", kind="decode", model="llama-3-8b", quant=False,
             rows=96, lo=1500, hi=4000),
        # routed experts, decode at the same load as above
        dict(name="mixtral decode 40 rows", kind="decode", model="mixtral-8x7b",
             quant=True, rows=40, lo=100, hi=700),
        # the mixed step of the chat load: a few users' new turns beside everybody
        # else's next token
        dict(name="mixed step fp8", kind="prompt", model="llama-3-8b", quant=True,
             rows=32, lo=100, hi=700, seqs=6, new_lo=48, new_hi=112, hist=600, adapters=0),
        # one prompt of ordinary length
        dict(name="prompt 2000 bf16", kind="prompt", model="llama-3-8b", quant=False,
             rows=0, lo=0, hi=0, seqs=1, new_lo=2000, new_hi=2000, hist=0, adapters=0),
        # a document that fills the step's token budget
        dict(name="prompt 8192 fp8", kind="prompt", model="llama-3-8b", quant=True,
             rows=0, lo=0, hi=0, seqs=1, new_lo=8192, new_hi=8192, hist=0, adapters=0),
        # routed experts, several prompts at once
        dict(name="mixtral prompts 2000", kind="prompt", model="mixtral-8x7b", quant=True,
             rows=0, lo=0, hi=0, seqs=3, new_lo=400, new_hi=900, hist=0, adapters=0),
        # four adapters over one base model, decode rows and new prompts
        dict(name="adapters step", kind="prompt", model="llama-3-8b", quant=False,
             rows=28, lo=100, hi=700, seqs=4, new_lo=20, new_hi=120, hist=0, adapters=4),
        # head size 256, window on every other layer, capped scores
        dict(name="gemma prompts 5000", kind="prompt", model="gemma2-2b", quant=False,
             rows=0, lo=0, hi=0, seqs=2, new_lo=900, new_hi=3900, hist=0, adapters=0),
        # a layer-list design: window attention with a sink, latent attention,
        # routed squared-ReLU experts
        dict(name="nugopel prompt 3000", kind="prompt", model="nugopel-2k", quant=False,
             rows=0, lo=0, hi=0, seqs=1, new_lo=3000, new_hi=3000, hist=0, adapters=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A decode step, a step with prompt portions, a step with adapters or a
    run of whole requests, at sizes spread over what the listed ones span."""
    kind = rng.choice(["decode"] * 5 + ["prompt"] * 6 + ["adapters", "chat"])
    if kind == "chat":
        lo = _log(rng, 16, 200)
        return dict(kind="chat", model="llama-3-8b", quant=rng.random() < 0.5,
                    rows=_log(rng, 4, 48), lo=lo, hi=lo + _log(rng, 1, 100),
                    new=rng.randint(4, 9))
    if kind == "decode":
        model = rng.choice(["llama-3-8b", "llama-3-8b", "mixtral-8x7b", "gemma2-2b",
                            "nugopel-2k"])
        rows = _log(rng, 1, 96)
        lo = _log(rng, 20, 2500)
        return dict(kind="decode", model=model,
                    quant=model in ("llama-3-8b", "mixtral-8x7b") and rng.random() < 0.6,
                    rows=rows, lo=lo, hi=lo + _log(rng, 1, 1500))
    if kind == "adapters":
        return dict(kind="prompt", model="llama-3-8b", quant=False, rows=_log(rng, 1, 48),
                    lo=50, hi=_log(rng, 60, 1500), seqs=rng.randint(0, 4), new_lo=5,
                    new_hi=_log(rng, 6, 300), hist=0, adapters=rng.randint(1, 5))
    model = rng.choice(["llama-3-8b", "llama-3-8b", "mixtral-8x7b", "gemma2-2b",
                        "nugopel-2k"])
    seqs = rng.choice([1, 1, 1, 2, 3, 6])
    longest = _log(rng, 17, 7000)
    if model != "llama-3-8b":
        longest = min(longest, 4400)
    per = max(4, longest // seqs)
    mixed = rng.random() < 0.4
    return dict(kind="prompt", model=model,
                quant=model in ("llama-3-8b", "mixtral-8x7b") and rng.random() < 0.6,
                rows=_log(rng, 1, 40) if mixed else 0, lo=50, hi=_log(rng, 60, 1000),
                seqs=seqs, new_lo=max(2, per * 2 // 3), new_hi=per,
                hist=_log(rng, 10, 1500) if rng.random() < 0.4 else 0, adapters=0)


def _lengths(case):
    """[(tokens in the cache, new tokens)], one-token rows first; a case's
    lengths are its own and do not depend on the seed."""
    rng = random.Random(repr(sorted((k, v) for k, v in case.items() if k != "name")))
    if case["kind"] == "chat":
        return [(0, rng.randint(case["lo"], case["hi"])) for _ in range(case["rows"])]
    got = [(rng.randint(case["lo"], case["hi"]), 1) for _ in range(case["rows"])]
    if case["kind"] == "prompt":
        for _ in range(case["seqs"]):
            hist = rng.randint(case["hist"] // 2, case["hist"])
            got.append((hist, rng.randint(case["new_lo"], case["new_hi"])))
    return got


def _arch(case):
    a = PRESETS[case["model"]]
    n = FAMILIES[case["model"]]
    if a.hybrid is not None:
        hy = dataclasses.replace(a.hybrid, layers=a.hybrid.layers[:n])
        return dataclasses.replace(a, num_hidden_layers=n, hybrid=hy)
    return dataclasses.replace(a, num_hidden_layers=n)


# -------------------------------------------------------------- their inputs
class _Source:
    """Random tensors by name, the same ones for the same seed."""

    def __init__(self, seed, device="cuda"):
        self.seed, self.device = seed, device
        self.g = torch.Generator(device=device)

    def normal(self, name, shape, std=1.0, mean=0.0):
        self.g.manual_seed(zlib.crc32(name.encode()) + 7919 * self.seed)
        x = torch.empty(shape, dtype=torch.bfloat16, device=self.device)
        return x.normal_(mean, std, generator=self.g)


def _tokens(case, seed):
    vocab = PRESETS[case["model"]].vocab_size
    rng = random.Random(seed * 31 + 5)
    return [[rng.randrange(10, vocab - 10) for _ in range(n)] for _, n in _lengths(case)]


def _tables(case, seed):
    """Cache blocks of every sequence, scattered over the pool, and its size."""
    need = [(c + n + BLOCK - 1) // BLOCK for c, n in _lengths(case)]
    ids = list(range(1, sum(need) + 1))
    random.Random(seed * 17 + 3).shuffle(ids)
    out, at = [], 0
    for n in need:
        out.append(ids[at : at + n])
        at += n
    return out, sum(need) + 1


def _weights(case, a, src):
    """(name, tensor) of the decoder in the layout it is served from: q, k and
    v stacked, gate and up stacked. Scores have unit variance; a branch is
    small beside what it is added to, as in trained stacks, and smaller where
    values are rounded to eight bits: two correct programs round a few values
    to different sides, and in stacks with large branches each layer would
    multiply that until little else is left."""
    H, I, V, D = a.hidden_size, a.intermediate_size, a.vocab_size, a.head_dim
    nq, nk = a.num_attention_heads * D, a.num_key_value_heads * D
    small = H ** -0.5 if a.scale_embeddings else 1.0
    branch = 0.06 if case["quant"] else 0.3
    embed = src.normal("embed", (V, H), small)
    yield "embed_tokens.weight", embed
    yield "norm", src.normal("norm", (H,), 0.1, 1.0)
    if not a.tie_word_embeddings:
        head = src.normal("head", (V, H), H ** -0.5)
        if case["kind"] == "chat":
            # a model that has learnt something: after a token the one that
            # follows it in the table stands out from the rest
            head = head + torch.roll(embed, 1, 0) * (8.5 / H)
        yield "lm_head.weight", head
    for i in range(a.num_hidden_layers):
        p = "layers.%d." % i
        names = ["input_layernorm", "post_attention_layernorm"]
        if a.post_norms:
            names += ["pre_feedforward_layernorm", "post_feedforward_layernorm"]
        for n in names:
            yield p + n, src.normal(p + n, (H,), 0.1, 1.0)
        yield (p + "self_attn.qkv_proj.weight",
               src.normal(p + "qkv", (nq + 2 * nk, H), H ** -0.5))
        yield p + "self_attn.o_proj.weight", src.normal(p + "o", (H, nq), branch * nq ** -0.5)
        if a.num_local_experts:
            yield p + "mlp.gate.weight", src.normal(p + "gate", (a.num_local_experts, H),
                                                    2.0 * H ** -0.5)
        for e in range(max(1, a.num_local_experts)):
            q = p + ("mlp.experts.%d." % e if a.num_local_experts else "mlp.")
            yield q + "gate_up_proj.weight", src.normal(q + "gu", (2 * I, H), H ** -0.5)
            yield q + "down_proj.weight", src.normal(q + "down", (H, I), branch * I ** -0.5)


def _nugopel_weights(a, src):
    """(name, tensor) under the names of the design's checkpoints."""
    W, V = a.hidden_size, a.vocab_size

    def mat(name, o, i, gain=1.0):
        return name, src.normal(name, (o, i), gain * i ** -0.5)

    def vec(name, n, center):
        return name, src.normal(name, (n,), 0.1, center)

    yield "embed", src.normal("embed", (V, W))
    yield mat("head", V, W)
    yield vec("final.norm", W, 0.0)
    for i, L in enumerate(a.hybrid.layers):
        p, m, f = "l%d." % i, L.mixer, L.mlp
        for n in ("norm1", "norm1b", "norm2", "norm2b"):
            yield vec(p + n, W, 0.0)
        H, D, Dv = m["heads"], m["dim"], m["vdim"]
        yield mat(p + "mix.q", H * D, W)
        yield mat(p + "mix.o", W, H * Dv)
        if L.type == "attention":
            G = m["kv_heads"]
            yield mat(p + "mix.k", G * D, W)
            yield mat(p + "mix.v", G * Dv, W)
            yield vec(p + "mix.q.norm", H * D, 1.0)
            yield vec(p + "mix.k.norm", G * D, 1.0)
        else:
            R = m["kv_rank"]
            yield mat(p + "mix.uk", H * D, R)
            yield mat(p + "mix.uv", H * Dv, R)
            yield mat(p + "mix.g", H * Dv, W)
            if m.get("kv_from") is None:
                yield mat(p + "mix.dkv", R, W)
                yield vec(p + "mix.dkv.norm", R, 1.0)
        ff = f["expert"]["ff"]
        yield mat(p + "mlp.router", f["router"]["experts"], W, 2.0)
        for e in list(range(f["router"]["experts"])) + ["shared"]:
            q = p + ("mlp.shared." if e == "shared" else "mlp.e%d." % e)
            yield mat(q + "up", ff, W)
            yield mat(q + "down", W, ff)


def prepare(case, seed):
    a, src = _arch(case), _Source(seed)
    tables, blocks = _tables(case, seed)
    lens = _lengths(case)
    name = case["model"] + ", %d layers" % a.num_hidden_layers
    PRESETS[name] = a
    longest = max(c + n for c, n in lens) + case.get("new", 0)
    if case["kind"] == "chat":
        blocks += 2 * case["rows"]
    eng = LLMEngine(EngineConfig(
        model=name, device="cuda", num_gpu_blocks=blocks, max_model_len=longest + BLOCK,
        max_num_seqs=max(64, case["rows"]), max_num_batched_tokens=8192,
        enable_prefix_caching=False))
    model = eng.runner.model
    with torch.no_grad():
        if a.hybrid is not None:
            model.load_named_tensors(_nugopel_weights(a, src))
        else:
            params = dict(model.named_parameters())
            for n, w in _weights(case, a, src):
                params[n].copy_(w)
        if case["quant"]:
            convert_to_fp8(model)
        caches = [c for c in eng.runner.kv_caches if c is not None]
        for i, layer in enumerate(caches):
            for j, t in enumerate(layer):
                t.copy_(src.normal("cache%d.%d" % (i, j), t.shape))
    toks = _tokens(case, seed)
    state = {"kind": case["kind"], "engine": eng, "tokens": toks,
             "kv": [t for layer in caches for t in layer if t.numel()]}
    if case["kind"] == "chat":
        state.update(new=case["new"], turn=0)
        return state
    for k in range(case.get("adapters", 0)):
        eng.load_lora(k + 1, None)
    rows, want = [], {}
    for i, ((c, n), t) in enumerate(zip(lens, toks)):
        lora = i % (case["adapters"] + 1) if case.get("adapters") else 0
        r = Request([10] * c + t, SamplingParams(), request_id="s%d" % i, lora_id=lora)
        r.block_table = tables[i]
        rows.append(ScheduledSeq(r, c, n))
        want[r.request_id] = [n - 1]
    if case["kind"] == "prompt":
        state["step"] = SchedulerOutput(decode=rows[: case["rows"]],
                                        prefill=rows[case["rows"] :], preempted=[])
        state["want"] = want
        return state
    # the engine's graphs are recorded for these many rows; idle ones write nothing
    idle = -len(rows) % (8 if len(rows) <= 48 else 16)
    for i in range(idle):
        r = Request([10], SamplingParams(), request_id="idle%d" % i)
        r.block_table = [0]
        rows.append(ScheduledSeq(r, 0, 1))
    fb = eng.runner.build_batch(SchedulerOutput(decode=rows, prefill=[], preempted=[]))
    fb.slot_mapping[case["rows"] :] = -1

    def forward():
        return model.compute_logits(model(fb))

    forward()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = forward()
    state.update(graph=graph, batch=fb, logits=logits[: case["rows"]])
    return state


def run(state):
    eng = state["engine"]
    if state["kind"] == "decode":
        state["graph"].replay()
        return {"logits": state["logits"], "kv": state["kv"]}
    if state["kind"] == "prompt":
        logits = eng.runner.forward_logits(state["step"], state["want"])
        return {"logits": logits, "kv": state["kv"]}
    state["turn"] += 1
    params = SamplingParams(max_tokens=state["new"], temperature=0.0, ignore_eos=True)
    ids = ["t%d-u%d" % (state["turn"], u) for u in range(len(state["tokens"]))]
    for rid, toks in zip(ids, state["tokens"]):
        eng.add_request(toks, params, request_id=rid)
    got = {rid: ([], []) for rid in ids}
    while eng.has_work():
        for o in eng.step():
            got[o.request_id][0].extend(o.new_token_ids)
            got[o.request_id][1].append(o.logprob)
    return {"tokens": torch.tensor([got[r][0] for r in ids]),
            "logprobs": torch.tensor([got[r][1] for r in ids])}


# ------------------------------------------------- what a pass cannot do without
def work(case):
    a, lens = _arch(case), _lengths(case)
    if case["kind"] == "chat":
        total = {"bytes": 0.0, "flops": 0.0}
        for parts in [lens] + [[(n + k, 1) for _, n in lens] for k in range(case["new"] - 1)]:
            w = _step_work(a, case, parts)
            total = {k: total[k] + w[k] for k in total}
        return total
    return _step_work(a, case, lens)


def _pairs(c, n, window):
    """Query-key pairs of n new tokens behind c old ones."""
    if not window:
        return n * c + n * (n + 1) / 2
    return sum(min(c + k + 1, window) for k in range(n))


def _keys(c, n, window):
    return min(c + n, window + n - 1) if window else c + n


def _step_work(a, case, lens):
    T, S, H = sum(n for _, n in lens), len(lens), a.hidden_size
    wb = 1 if case["quant"] else 2
    b = T * H * 2 + a.vocab_size * H * (2 if a.tie_word_embeddings or a.hybrid else wb) \
        + 4 * S * a.vocab_size
    f = 2.0 * S * a.vocab_size * H

    def layer(fixed, experts, top, expert, score, value, cached, window):
        """fixed/expert: weights; score/value: multiplied per query-key pair;
        cached: bytes kept per token."""
        nonlocal b, f
        hit = experts * (1 - (1 - top / experts) ** T) if experts else 0
        b += fixed * wb + hit * expert * wb
        f += 2.0 * T * (fixed + top * expert)
        b += sum(_keys(c, n, window) for c, n in lens) * cached
        f += 2.0 * (score + value) * sum(_pairs(c, n, window) for c, n in lens)

    if a.hybrid is None:
        D, nq, nk = a.head_dim, a.num_attention_heads, a.num_key_value_heads
        mlp = 3 * H * a.intermediate_size
        for i in range(a.num_hidden_layers):
            win = a.sliding_window if a.sliding_window_pattern != "even" or i % 2 == 0 else 0
            fixed = H * (nq + 2 * nk) * D + nq * D * H
            E = a.num_local_experts
            layer(fixed if E else fixed + mlp, E, a.num_experts_per_tok if E else 0, mlp,
                  nq * D, nq * D, 4 * nk * D, win)
            if case.get("adapters"):
                io = H + (nq + 2 * nk) * D + nq * D + H + H + 2 * a.intermediate_size \
                    + a.intermediate_size + H
                b += 2 * RANK * io * case["adapters"]
                f += 2.0 * T * RANK * io * case["adapters"] / (case["adapters"] + 1)
        return {"bytes": float(b), "flops": float(f)}
    for L in a.hybrid.layers:
        m, fm = L.mixer, L.mlp
        E, ff = fm["router"]["experts"], fm["expert"]["ff"]
        hd, hv = m["heads"] * m["dim"], m["heads"] * m["vdim"]
        fixed = H * hd + H * hv + 2 * H * ff + H * E
        if L.type == "attention":
            g = m["kv_heads"] * (m["dim"] + m["vdim"])
            layer(fixed + H * g, E, fm["router"]["top"], 2 * H * ff, hd, hv, 2 * g,
                  m["mask"]["size"])
        else:
            R = m["kv_rank"]
            own = m.get("kv_from") is None
            layer(fixed + H * hv + R * (hd + hv) + (H * R if own else 0), E,
                  fm["router"]["top"], 2 * H * ff, m["heads"] * R, m["heads"] * R, 2 * R, 0)
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    # four times the distance from the 64-bit results, at most what counts as
    # the same; a token may differ where two candidates all but tie, and routed
    # models move a token to another expert where two scores all but tie
    if case["kind"] == "chat":
        return {"rel": 0.03, "max": 0.6, "differ": 0.01}
    if case["quant"] or case["model"] in ("mixtral-8x7b", "nugopel-2k"):
        return {"rel": 0.03, "max": 0.9}
    return {"rel": 0.02, "max": 0.3}


# --------------------------------------------------------- the same in 64 bits
def _rms(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _fp8_rows(x):
    """x rounded to eight bits with one scale a row, back in 64 bits."""
    s = (x.abs().amax(-1, keepdim=True) / 448.0).clamp_min(1e-30)
    return (x / s).clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn).double() * s


def _frequencies(D, base, sc, dims=None):
    dims = dims or D
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)
    if not sc:
        return f
    lo, hi = sc.get("low_freq_factor", sc.get("low")), sc.get("high_freq_factor", sc.get("high"))
    orig = sc.get("original_max_position_embeddings", sc.get("original"))
    turns = orig * f / (2 * math.pi)  # whole turns over the original length
    s = ((turns - lo) / (hi - lo)).clamp(0.0, 1.0)
    return (1 - s) * f / sc["factor"] + s * f


def _rotate(x, pos, f):
    """x [n, heads, D]: dimension i of the first 2 len(f) turns with i + len(f)."""
    ang = pos[:, None, None].double() * f
    c, s, h = ang.cos(), ang.sin(), len(f)
    u, v = x[..., :h], x[..., h : 2 * h]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * h :]], -1)


def _attend(q, k, v, c, scale, window=0, cap=0.0, sink=False):
    """q [n, heads, D] behind c old tokens, k/v [c + n, groups, D]."""
    n, H, _ = q.shape
    rep = H // k.shape[1]
    out = torch.empty(n, H, v.shape[-1], dtype=torch.float64, device=q.device)
    j = torch.arange(k.shape[0], device=q.device)
    step = max(1, int(2 ** 27 // max(1, k.shape[0])))
    for h in range(H):
        kk, vv = k[:, h // rep], v[:, h // rep]
        for lo in range(0, n, step):
            i = torch.arange(c + lo, c + min(n, lo + step), device=q.device)[:, None]
            s = q[lo : lo + step, h] @ kk.T * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            see = j[None] <= i
            if window:
                see &= i - j[None] < window
            s = s.masked_fill(~see, -math.inf)
            if sink:
                s = torch.cat([s, torch.zeros_like(s[:, :1])], 1)
                out[lo : lo + step, h] = torch.softmax(s, -1)[:, :-1] @ vv
            else:
                out[lo : lo + step, h] = torch.softmax(s, -1) @ vv
    return out


class _Cache:
    """The key and value rows of a layer, by sequence."""

    def __init__(self, src, name, tables, blocks, heads, dim):
        self.t = src.normal(name, (blocks, heads, BLOCK, dim))
        self.tables = tables

    def old(self, i, c):
        if c == 0:
            return self.t[:0, :, 0].double()
        ids = torch.tensor(self.tables[i], device=self.t.device)
        return self.t[ids].transpose(1, 2).flatten(0, 1)[:c].double()

    def put(self, i, c, rows):
        at = torch.arange(c, c + rows.shape[0], device=rows.device)
        ids = torch.tensor(self.tables[i], device=rows.device)[at // BLOCK]
        self.t[ids, :, at % BLOCK] = rows


def _exact_llama(case, a, seed, lens, toks, tables, blocks, every=False):
    """Logits of each sequence's last token (of all tokens with every=True) and
    the caches after the step."""
    src = _Source(seed)
    W = dict(_weights(case, a, src))
    x = W["embed_tokens.weight"][torch.tensor(sum(toks, []), device="cuda")].double()
    if a.scale_embeddings:
        x = x * a.hidden_size ** 0.5
    D, nq, nk = a.head_dim, a.num_attention_heads, a.num_key_value_heads
    f = _frequencies(D, a.rope_theta, a.rope_scaling)
    pos = torch.cat([torch.arange(c, c + n, device="cuda") for c, n in lens])
    scale = (a.query_pre_attn_scalar or D) ** -0.5
    q8 = _fp8_rows if case["quant"] else (lambda t: t)
    seq = []  # the adapter of every token
    if case.get("adapters"):
        for i, (_, n) in enumerate(lens):
            seq += [i % (case["adapters"] + 1)] * n
        seq = torch.tensor(seq, device="cuda")
    adapters = _adapters(case, a)

    def weight(name):
        w = W[name].double()
        if case["quant"]:
            s = (W[name].float().abs().amax(1, keepdim=True).clamp_min(1e-6) / 448.0)
            w = (W[name].float() / s).clamp(-448, 448).to(torch.float8_e4m3fn).double() * s
        return w

    def lin(t, name, target=None, layer=0):
        y = q8(t) @ weight(name).T
        for k, sets in enumerate(adapters):
            A, B = sets[target][layer] if target else (None, None)
            if target:
                on = (seq == k + 1)[:, None].double()
                y += on * (t @ A.double().T @ B.double().T) * (2.0 / RANK)
        return y

    def act(t):
        g, u = t.chunk(2, -1)
        if a.hidden_act == "gelu_pytorch_tanh":
            return torch.nn.functional.gelu(g, approximate="tanh") * u
        return torch.nn.functional.silu(g) * u

    def mlp(t, p, i):
        if not a.num_local_experts:
            h = act(lin(t, p + "mlp.gate_up_proj.weight", "gate_up", i))
            return lin(h, p + "mlp.down_proj.weight", "down", i)
        z = t @ W[p + "mlp.gate.weight"].double().T
        top, idx = z.topk(a.num_experts_per_tok, -1)
        wts = torch.softmax(top, -1)
        y = torch.zeros_like(t)
        for e in range(a.num_local_experts):
            on = (wts * (idx == e)).sum(-1)
            at = on.nonzero()[:, 0]
            q = p + "mlp.experts.%d." % e
            h = act(lin(t[at], q + "gate_up_proj.weight"))
            y[at] += on[at, None] * lin(h, q + "down_proj.weight")
        return y

    kv = []
    for i in range(a.num_hidden_layers):
        p = "layers.%d." % i
        win = a.sliding_window if a.sliding_window_pattern != "even" or i % 2 == 0 else 0
        norm = lambda t, n: _rms(t, W[p + n].double(), a.rms_norm_eps)  # noqa: E731
        h = lin(norm(x, "input_layernorm"), p + "self_attn.qkv_proj.weight", "qkv", i)
        q, k, v = h.split([nq * D, nk * D, nk * D], -1)
        q = _rotate(q.unflatten(-1, (nq, D)), pos, f)
        k, v = _rotate(k.unflatten(-1, (nk, D)), pos, f), v.unflatten(-1, (nk, D))
        ks = _Cache(src, "cache%d.0" % i, tables, blocks, nk, D)
        vs = _Cache(src, "cache%d.1" % i, tables, blocks, nk, D)
        o, at = [], 0
        for s, (c, n) in enumerate(lens):
            kk = torch.cat([ks.old(s, c), k[at : at + n]]) if c else k[at : at + n]
            vv = torch.cat([vs.old(s, c), v[at : at + n]]) if c else v[at : at + n]
            o.append(_attend(q[at : at + n], kk, vv, c, scale, win, a.attn_logit_softcap))
            at += n
        if tables is not None:
            at = 0
            ks.t, vs.t = ks.t.double(), vs.t.double()
            for s, (c, n) in enumerate(lens):
                ks.put(s, c, k[at : at + n])
                vs.put(s, c, v[at : at + n])
                at += n
            kv += [ks.t, vs.t] if not every else []
        y = lin(torch.cat(o).flatten(1), p + "self_attn.o_proj.weight", "o", i)
        if a.post_norms:
            x = x + norm(y, "post_attention_layernorm")
            y = mlp(norm(x, "pre_feedforward_layernorm"), p, i)
            x = x + norm(y, "post_feedforward_layernorm")
        else:
            x = x + y
            x = x + mlp(norm(x, "post_attention_layernorm"), p, i)
    x = _rms(x, W["norm"].double(), a.rms_norm_eps)
    if not every:
        x = x[torch.tensor([n for _, n in lens], device="cuda").cumsum(0) - 1]
    if a.tie_word_embeddings:
        logits = x @ W["embed_tokens.weight"].double().T
    else:
        logits = q8(x) @ weight("lm_head.weight").T
    if a.final_logit_softcap:
        logits = a.final_logit_softcap * torch.tanh(logits / a.final_logit_softcap)
    return logits, kv


def _adapters(case, a):
    """The adapters load_lora makes without files: [{target: [(A, B) by layer]}]."""
    H, I = a.hidden_size, a.intermediate_size
    nq, nk = a.num_attention_heads * a.head_dim, a.num_key_value_heads * a.head_dim
    out = []
    for k in range(case.get("adapters", 0)):
        g = torch.Generator().manual_seed(k + 1)
        sets = {"qkv": [], "o": [], "gate_up": [], "down": []}
        for _ in range(a.num_hidden_layers):
            for t, i, o in (("qkv", H, nq + 2 * nk), ("o", nq, H), ("gate_up", H, 2 * I),
                            ("down", I, H)):
                A = torch.randn(RANK, i, generator=g) * 0.05
                B = torch.randn(o, RANK, generator=g) * 0.5
                sets[t].append((A.bfloat16().cuda(), B.bfloat16().cuda()))
        out.append(sets)
    return out


def _exact_nugopel(case, a, seed, lens, toks, tables, blocks):
    src = _Source(seed)
    W = dict(_nugopel_weights(a, src))
    dbl = lambda n: W[n].double()  # noqa: E731
    eps = a.hybrid.norm_eps
    x = W["embed"][torch.tensor(sum(toks, []), device="cuda")].double()
    pos = torch.cat([torch.arange(c, c + n, device="cuda") for c, n in lens])
    caches, slot = {}, 0  # layer -> its rows by sequence
    for i, L in enumerate(a.hybrid.layers):
        p, m, fm = "l%d." % i, L.mixer, L.mlp
        norm = lambda t, n: _rms(t, 1 + dbl(p + n), eps)  # noqa: E731
        h = norm(x, "norm1")
        H, D, Dv = m["heads"], m["dim"], m["vdim"]
        q, o, at = h @ dbl(p + "mix.q").T, [], 0
        if L.type == "attention":
            G, rot = m["kv_heads"], m["rot"]
            f = _frequencies(D, rot["base"], rot["scaling"], rot["dims"])
            q = _rotate(_rms(q, dbl(p + "mix.q.norm"), eps).unflatten(-1, (H, D)), pos, f)
            k = _rms(h @ dbl(p + "mix.k").T, dbl(p + "mix.k.norm"), eps)
            k = _rotate(k.unflatten(-1, (G, D)), pos, f)
            v = (h @ dbl(p + "mix.v").T).unflatten(-1, (G, Dv))
            ks = _Cache(src, "cache%d.0" % slot, tables, blocks, G, D)
            vs = _Cache(src, "cache%d.1" % slot, tables, blocks, G, Dv)
            slot += 1
            for s, (c, n) in enumerate(lens):
                o.append(_attend(q[at : at + n], torch.cat([ks.old(s, c), k[at : at + n]]),
                                 torch.cat([vs.old(s, c), v[at : at + n]]), c, m["scale"],
                                 m["mask"]["size"], sink=True))
                at += n
            y = torch.cat(o).flatten(1)
        else:
            R = m["kv_rank"]
            if m.get("kv_from") is None:
                new = _rms(h @ dbl(p + "mix.dkv").T, dbl(p + "mix.dkv.norm"), eps)
                cs = _Cache(src, "cache%d.0" % slot, tables, blocks, 1, R)
                slot += 1
                caches[i] = []
                for s, (c, n) in enumerate(lens):
                    caches[i].append(torch.cat([cs.old(s, c)[:, 0], new[at : at + n]]))
                    at += n
            q = q.unflatten(-1, (H, D))
            uk, uv, at = dbl(p + "mix.uk"), dbl(p + "mix.uv"), 0
            for s, (c, n) in enumerate(lens):
                rows = caches[i if m.get("kv_from") is None else m["kv_from"]][s]
                o.append(_attend(q[at : at + n], (rows @ uk.T).unflatten(-1, (H, D)),
                                 (rows @ uv.T).unflatten(-1, (H, Dv)), c, m["scale"]))
                at += n
            y = torch.cat(o).flatten(1) * torch.sigmoid(h @ dbl(p + "mix.g").T)
        x = x + norm(y @ dbl(p + "mix.o").T, "norm1b")
        h = norm(x, "norm2")

        def expert(t, q):
            return torch.relu(t @ dbl(q + "up").T) ** 2 @ dbl(q + "down").T

        z, idx = (h @ dbl(p + "mlp.router").T).topk(fm["router"]["top"], -1)
        wts = torch.softmax(z, -1)
        y = expert(h, p + "mlp.shared.")
        for e in range(fm["router"]["experts"]):
            on = (wts * (idx == e)).sum(-1)
            at = on.nonzero()[:, 0]
            y[at] += on[at, None] * expert(h[at], p + "mlp.e%d." % e)
        x = x + norm(y, "norm2b")
    x = _rms(x, 1 + dbl("final.norm"), eps)
    x = x[torch.tensor([n for _, n in lens], device="cuda").cumsum(0) - 1]
    return x @ dbl("head").T


@torch.no_grad()
def exact(case, seed):
    """What run() returns, in 64 bits. Rounding to eight bits is part of what a
    quantised model computes and stays; nothing else is rounded."""
    a, lens, toks = _arch(case), _lengths(case), _tokens(case, seed)
    tables, blocks = _tables(case, seed)
    if a.hybrid is not None:
        return {"logits": _exact_nugopel(case, a, seed, lens, toks, tables, blocks), "kv": None}
    if case["kind"] != "chat":
        logits, kv = _exact_llama(case, a, seed, lens, toks, tables, blocks)
        return {"logits": logits, "kv": kv if case["kind"] == "prompt" else None}
    # follow the most likely token; a guess that proves wrong is replaced and
    # the sequences are run again
    new, V = case["new"], a.vocab_size
    full = [list(t) + [(t[-1] + k + 1) % V for k in range(new - 1)] for t in toks]
    for _ in range(new + 1):
        wrong, best, logp, at = False, [], [], 0
        logits, _ = _exact_llama(case, a, seed, [(0, len(t)) for t in full], full, None, 1,
                                 every=True)
        for t, whole in zip(toks, full):
            rows = logits[at + len(t) - 1 : at + len(whole)]
            at += len(whole)
            pick = rows.argmax(-1)
            logp.append(torch.log_softmax(rows, -1).gather(1, pick[:, None])[:, 0])
            best.append(pick)
            for k in range(new - 1):
                if whole[len(t) + k] != int(pick[k]):
                    whole[len(t) + k] = int(pick[k])
                    whole[len(t) + k + 1 :] = [(int(pick[k]) + m + 1) % V
                                               for m in range(new - 2 - k)]
                    wrong = True
                    break
        if not wrong:
            break
    return {"tokens": torch.stack(best), "logprobs": torch.stack(logp).float().double()}
