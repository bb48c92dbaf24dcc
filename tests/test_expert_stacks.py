"""The experts' stacked weights of MoEMLP as part of the module: what keeps them
alive, and what becomes of them when the module is moved, copied or loaded."""
import copy
import pickle
import weakref

import torch

from kubeai_amd.engine import quant
from kubeai_amd.models.config import PRESETS
from kubeai_amd.models.llama import LlamaForCausalLM, MoEMLP


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


def _mixture(dtype=torch.float32):
    torch.manual_seed(0)
    cfg = PRESETS["mixtral-tiny"]
    return MoEMLP(cfg).to(dtype), torch.randn(5, cfg.hidden_size, dtype=dtype)


def _stacked(m):
    return all(m._stack(p, "weight") is not None for p in ("gate_up_proj", "down_proj"))


def test_moved_copied_and_loaded_mixtures_stay_stacked():
    m, x = _mixture()
    assert _stacked(m)
    want = m(x)
    params = [id(p) for p in m.parameters()]
    old = weakref.ref(m._stacks["down_proj", "weight"])
    m.double()
    assert _stacked(m) and old() is None and [id(p) for p in m.parameters()] == params
    m.float()
    assert _stacked(m) and torch.equal(m(x), want)

    for other in (copy.deepcopy(m), pickle.loads(pickle.dumps(m))):
        assert _stacked(other) and torch.equal(other(x), want)
        with torch.no_grad():  # storage of its own
            other.experts[0].down_proj.weight.zero_()
        assert torch.equal(m(x), want) and not torch.equal(other(x), want)

    with torch.device("meta"):
        empty = MoEMLP(PRESETS["mixtral-tiny"])
    empty.load_state_dict({k: v.clone() for k, v in m.state_dict().items()}, assign=True)
    assert _stacked(empty) and torch.equal(empty(x), want)
    with torch.device("meta"):
        empty = MoEMLP(PRESETS["mixtral-tiny"])
    empty.to_empty(device="cpu").load_state_dict(m.state_dict())
    assert _stacked(empty) and torch.equal(empty(x), want)
    holder = torch.nn.Sequential(MoEMLP(PRESETS["mixtral-tiny"]))
    holder.load_state_dict({"0." + k: v for k, v in m.state_dict().items()})
    assert _stacked(holder[0]) and torch.equal(holder(x), want)


def test_a_replaced_weight_lets_the_stack_go():
    m, x = _mixture()
    old = weakref.ref(m._stacks["down_proj", "weight"])
    for e in m.experts:
        e.down_proj.weight = torch.nn.Parameter(e.down_proj.weight.detach() * 2)
    assert m._stack("down_proj", "weight") is None and old() is None
    want = m(x)
    m.stack_experts()
    assert _stacked(m) and torch.equal(m(x), want)
    with torch.inference_mode():
        m.stack_experts()
    m(x.clone().requires_grad_()).sum().backward()  # (ordinary tensors all the same)
    assert m.experts[0].down_proj.weight.grad is not None
    m.experts[1].down_proj = torch.nn.Linear(m.experts[1].down_proj.in_features, x.shape[1],
                                             bias=False, dtype=torch.float64)
    m.stack_experts()  # experts of different types are not stacked
    assert m._stack("down_proj", "weight") is None
    assert m._stack("gate_up_proj", "weight") is not None
