"""The rows of a large step's experts with the shared expert among them."""
import pytest
import torch

from kubeai_amd import ops
from kubeai_amd.models.mixers import RoutedSquaredReluMoE
from kubeai_amd.ops import seq as sops

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("T,E,top", [(1, 1, 1), (7, 3, 2), (257, 8, 2), (1025, 5, 3),
                                     (2048, 70, 1)])
def test_one_more_expert_has_every_token(device, T, E, top):
    """The same rows, places and counts as when each token chooses it itself."""
    g = torch.Generator().manual_seed(T)
    idx = torch.rand(T, E, generator=g).argsort(1)[:, :top].int()
    w = torch.rand(T, top, generator=g)
    got = sops.expert_order(idx.to(device), w.to(device), E, every=True)
    more = torch.cat([idx, torch.full((T, 1), E, dtype=torch.int32)], 1)
    want = sops.expert_order(more, torch.cat([w, torch.ones(T, 1)], 1), E + 1)
    for a, b in zip(got, want):
        assert a.shape == b.shape and torch.equal(a.cpu(), b)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [257, 300, 1024, 3000])
@pytest.mark.parametrize("W,E,top,ff,shared", [(256, 4, 2, 128, 128), (512, 8, 2, 448, 448),
                                               (256, 4, 1, 128, 64), (256, 3, 2, 80, 80)])
def test_mixture_with_a_shared_expert(T, W, E, top, ff, shared):
    """Shared experts of the others' size, of another one, and of rows that the tiled
    product does not take, against fp32."""
    torch.manual_seed(T)
    moe = RoutedSquaredReluMoE(W, E, top, ff, shared).to("cuda", torch.bfloat16)
    moe.router.data = moe.router.data.float()
    h = torch.randn(T, W, device="cuda").bfloat16()
    got = moe(h).float()
    up, down, x = moe.up.weight.float(), moe.down.weight.float(), h.float()
    dense, _, _ = sops.router_topk(x @ moe.router.t(), top)
    a = torch.relu(x @ up.t()).square()
    a[:, : E * ff] *= dense.repeat_interleave(ff, 1)
    want = a @ down.t()
    # three roundings to bf16 in a row (2^-9 each, at most), of independent signs
    assert (got - want).norm() / want.norm() < 5e-3
    assert ops.have_hip_ext()
