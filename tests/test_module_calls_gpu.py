"""Modules whose calls someone else waits for: forward hooks see every call and
get tensors, also where the layers would hand products on unadded (few rows)."""
import pytest
import torch

import kubeai_amd.ops as ops
from kubeai_amd.engine import EngineConfig, LLMEngine
from kubeai_amd.engine.batch import ForwardBatch
from kubeai_amd.engine.quant import Fp8Linear, convert_to_fp8
from kubeai_amd.models.config import PRESETS
from kubeai_amd.models.llama import MoEMLP

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _step(model_name, fp8):
    torch.manual_seed(0)
    eng = LLMEngine(EngineConfig(model=model_name, device=DEV, num_gpu_blocks=32,
                                 max_model_len=128))
    model = eng.runner.model
    if fp8:
        convert_to_fp8(model)
    T = 8
    fb = ForwardBatch(
        input_ids=torch.arange(20, 20 + T, dtype=torch.int32, device=DEV),
        positions=torch.zeros(T, dtype=torch.int32, device=DEV),
        slot_mapping=torch.arange(16, 16 * (T + 1), 16, device=DEV), n_decode=T,
        decode_block_tables=torch.arange(1, T + 1, dtype=torch.int32, device=DEV).view(T, 1),
        decode_seq_lens=torch.ones(T, dtype=torch.int32, device=DEV), n_prefill=0,
        prefill_query_start_loc=None, prefill_seq_lens=None, prefill_block_tables=None,
        logits_indices=torch.arange(T, device=DEV))
    return model, fb


@pytest.mark.parametrize("name", ["llama-tiny", "gemma2-tiny"])
def test_hooks_see_tensors(name):
    model, fb = _step(name, False)
    want = model(fb).float()
    seen = []
    for part, mod in model.named_modules():
        if part.startswith("layers."):
            mod.register_forward_hook(
                lambda m, args, out, part=part: seen.append((part, args, out)))
    got = model(fb).float()
    # sums of another product's parts: one rounding here and there
    assert (got - want).norm() < 0.02 * want.norm()
    names = {p for p, _, _ in seen}
    for i in range(len(model.layers)):
        for part in ("", ".self_attn", ".self_attn.qkv_proj", ".self_attn.o_proj", ".mlp",
                     ".mlp.gate_up_proj", ".mlp.down_proj"):
            assert "layers.%d%s" % (i, part) in names
    for _, args, out in seen:
        for t in list(args) + (list(out) if isinstance(out, tuple) else [out]):
            assert not isinstance(t, ops.ProductSums)


@pytest.mark.parametrize("fp8", [False, True])
def test_a_layer_called_by_itself_returns_tensors(fp8):
    model, fb = _step("llama-tiny", fp8)
    layer = model.layers[0]
    with torch.inference_mode():
        x = model.embed_tokens(fb.input_ids.long())
        out = layer(x, None, fb, model.kv_caches[0], model.cos_sin)
        assert all(type(t) is torch.Tensor for t in out)
        layer.register_forward_hook(lambda m, args, o: None)
        model(fb)


def test_fp8_modules_put_in_by_others():
    """They get the calls that Fp8Linear and MLP got: forward_quantized(rows,
    scales) for a projection, one argument for a feed-forward module."""
    model, fb = _step("llama-tiny", True)
    with torch.inference_mode():
        want = model(fb).float()
        layer = model.layers[0]
        calls = []

        class Watched(Fp8Linear):
            def forward_quantized(self, xq, x_scale):
                calls.append("derived")
                return super().forward_quantized(xq, x_scale)

        class Other(torch.nn.Module):
            def __init__(self, lin):
                super().__init__()
                self.lin = lin

            def forward_quantized(self, xq, x_scale):
                calls.append("other")
                return self.lin.forward_quantized(xq, x_scale)

        class Feed(torch.nn.Module):
            def __init__(self, mlp):
                super().__init__()
                self.mlp = mlp

            def forward(self, x):
                calls.append("feed")
                return self.mlp(x)

        layer.mlp.down_proj.__class__ = Watched
        layer.self_attn.o_proj = Other(layer.self_attn.o_proj)
        layer.mlp = Feed(layer.mlp)
        got = model(fb).float()
    assert calls == ["other", "feed", "derived"]
    # sums of another product's parts: one rounding here and there
    assert (got - want).norm() < 0.02 * want.norm()


def test_expert_hooks():
    with torch.device(DEV):
        m = MoEMLP(PRESETS["mixtral-tiny"]).bfloat16()
    calls = []
    for T in (6, 300):
        x = torch.randn(T, m.gate.in_features, device=DEV, dtype=torch.bfloat16)
        with torch.inference_mode():
            want = m(x).float()
            h = m.experts[1].down_proj.register_forward_hook(lambda *a: calls.append(T))
            got = m(x).float()
            h.remove()
        assert T in calls
        # the per-expert route rounds weights and partial sums to bf16
        assert (got - want).norm() < 0.02 * want.norm()
