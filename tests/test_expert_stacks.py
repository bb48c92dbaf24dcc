"""The experts' stacked weights of MoEMLP as part of the module: what keeps them
alive, and what becomes of them when the module is moved, copied or loaded."""
import weakref

import torch

from kubeai_amd.engine import quant
from kubeai_amd.models.config import PRESETS
from kubeai_amd.models.llama import LlamaForCausalLM


def test_conversion_frees_each_layers_weights(monkeypatch):
    """When a layer's experts are converted, no earlier layer's weights are left."""
    model = LlamaForCausalLM(PRESETS["mixtral-tiny"], dtype=torch.bfloat16)
    stacks = [weakref.ref(layer.mlp._stacks["gate_up_proj", "weight"]) for layer in model.layers]
    alive = []
    plain = quant.Fp8Linear.__init__

    def init(self, *args):
        alive.append(sum(r() is not None for r in stacks))
        plain(self, *args)

    monkeypatch.setattr(quant.Fp8Linear, "__init__", init)
    n = quant.convert_to_fp8(model)
    layers = len(stacks)
    assert layers >= 2 and n == len(alive) and 1 in alive and alive == sorted(alive, reverse=True)
    assert not any(r() is not None for r in stacks)
    for layer in model.layers:
        for proj in ("gate_up_proj", "down_proj"):
            assert layer.mlp._stack(proj, "weight_fp8") is not None
            assert layer.mlp._stack(proj, "weight_scale") is not None
